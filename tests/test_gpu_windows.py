"""Top-K windows of 65 to 1024 over rows that have fewer finite logits than the window, or hardly more (GPU): the oracle's
results, from the window kernels and not from the sort."""
import numpy as np
import pytest

import parity_util
from ncnn_moe_runtime_amd import hip_sampler, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("vocab", [1030, 16411, 100003])
def test_windows_over_few_finite_logits(dtype, vocab):
    rng = np.random.default_rng(vocab)
    finite = [0, 1, 2, 40, 64, 65, 100, 199, 200, 201, 500, 999, 1000, 1001, 1024]
    rows = 2 * len(finite)
    print("[case] few finite logits, %d x %d %s" % (rows, vocab, dtype), flush=True)
    logits = np.full((rows, vocab), -np.inf, dtype=np.float32)
    for i, row in enumerate(logits):
        at = rng.choice(vocab, finite[i // 2], replace=False)
        row[at] = rng.standard_normal(len(at)) * 2
    logits[3::8, 5] = np.nan
    logits[7, 9] = np.inf
    params = hip_sampler.make_params(rows, 0.9, 0, 0.97, 0.0)
    params["top_k"] = np.where(np.arange(rows) % 2 == 0, 200, 1000)
    params["min_p"][5::7] = np.float32(0.01)
    uniforms = rng.random(rows, dtype=np.float32)
    data = workloads.float32_to_bf16_bits(logits) if dtype == "bf16" else logits
    cpu = parity_util.run_oracle(data, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(data)
        gpu = sampler.sample(params, uniforms)
        again = sampler.sample(params, uniforms)
    parity_util.assert_results_match(gpu, cpu, dtype, "few finite logits")
    assert gpu.tobytes() == again.tobytes()
    assert (gpu["flags"] & hip_sampler.FLAG_GENERAL_PATH == 0).all()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("kind", ["halves", "sixteenths", "one far above", "all equal"])
def test_windows_over_many_neighbours(kind, dtype):
    """Hundreds and thousands of candidates of one value, or next to each other because another lies far above them."""
    rng = np.random.default_rng(7)
    rows, vocab = 12, 50021
    print("[case] many neighbours, %s %s" % (kind, dtype), flush=True)
    base = rng.standard_normal((rows, vocab)) * 2.5
    logits = {"halves": np.round(base * 2) / 2, "sixteenths": np.round(base * 16) / 16, "one far above": base, "all equal": np.full((rows, vocab), 1.5)}[kind].astype(np.float32)
    if kind == "one far above":
        logits[np.arange(rows), rng.integers(0, vocab, rows)] = 1e5
    if kind == "all equal":
        logits[:, rng.choice(vocab, vocab - 3000, replace=False)] = -np.inf  # (more than 4,096 candidates go to the sort)
    uniforms = rng.random(rows, dtype=np.float32)
    data = workloads.float32_to_bf16_bits(logits) if dtype == "bf16" else logits
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(data)
        for top_k, top_p in ((65, 1.0), (200, 0.95), (1000, 1.0), (1024, 0.9)):
            params = hip_sampler.make_params(rows, 1.0, top_k, top_p, 0.0)
            cpu = parity_util.run_oracle(data, params, uniforms)
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, dtype, "%s top_k %d" % (kind, top_k))
