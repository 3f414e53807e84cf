"""Top-K windows of 65 to 1024 over rows that have fewer finite logits than the window, or hardly more (GPU): the oracle's
results, from the window kernels and not from the sort."""
import numpy as np
import pytest
import torch  # in front of the sampler's library: both then share the HIP runtime that torch brings along

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


@pytest.mark.parametrize("spread,rounded", [(0.0, 0), (0.05, 0), (1.0, 0), (2.5, 0), (2.5, 16), (8.0, 0)])
def test_sums_over_the_edges_of_their_chunks(spread, rounded):
    """Windows that end at and next to the chunks of 64 terms, the 32 terms added at a time and the four terms of a lane, the draw and the Top-P
    stop anywhere among them.  (spread 0.05: the sums leave a binade inside most chunks; 8: most terms are below half an ulp.)"""
    rng = np.random.default_rng(int(spread * 100) + rounded)
    windows = [65, 66, 95, 96, 97, 127, 128, 129, 130, 131, 132, 133, 191, 192, 193, 255, 256, 257, 320, 511, 512, 513, 575, 576, 577, 641, 1000, 1023, 1024]
    rows, vocab = 4 * len(windows), 5003
    print("[case] chunk edges, spread %g" % spread, flush=True)
    logits = rng.standard_normal((rows, vocab)) * spread
    if rounded:
        logits = np.round(logits * rounded) / rounded
    logits = (logits + np.linspace(0, 0.5, vocab) * (spread == 0.0)).astype(np.float32)
    params = hip_sampler.make_params(rows, 1.0, 0, 1.0, 0.0)
    params["top_k"] = np.repeat(np.array(windows, dtype=np.uint32), 4)
    params["top_p"] = rng.choice(np.array([1.0, 0.9999, 0.97, 0.6, 0.1], dtype=np.float32), rows)
    params["min_p"][::5] = np.float32(0.02)
    uniforms = rng.random(rows, dtype=np.float32)
    uniforms[::7] = np.float32(1.0 - 2.0 ** -24)
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(logits)
        parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "chunk edges, spread %g" % spread)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("rows,vocab", [(1, 131), (7, 2051), (3, 100003), (130, 33001), (130, 65537), (256, 4099), (257, 4099)])
def test_windows_over_the_edges_of_parts(rows, vocab, dtype):
    """Rows side by side in memory, so that they begin at every alignment: one part a row and sixteen, a part of one batch of loads and of
    more, calls of one launch and of two; tokens and NaNs at the rows' ends, where a vector holds a neighbour's."""
    rng = np.random.default_rng(rows + vocab)
    print("[case] edges of parts, %d x %d %s" % (rows, vocab, dtype), flush=True)
    logits = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
    logits[0::3, 0] = 9.0
    logits[1::3, vocab - 1] = 9.5
    logits[2::5, vocab - 1] = np.nan
    logits[3::5, 0] = np.nan
    logits[4::7, 1:-1] = np.sort(logits[4::7, 1:-1])
    params = hip_sampler.make_params(rows, 0.9, 0, 0.97, 0.0)
    params["top_k"] = rng.choice([65, 100, 300, 1000], rows)
    params["min_p"][5::7] = np.float32(0.01)
    uniforms = rng.random(rows, dtype=np.float32)
    data = workloads.float32_to_bf16_bits(logits) if dtype == "bf16" else logits
    cpu = parity_util.run_oracle(data, params, uniforms)
    device = [torch.from_numpy(x).cuda() for x in (data.view(np.int16) if dtype == "bf16" else data, params.view(np.uint8), uniforms)]
    results = torch.zeros(rows * 16, dtype=torch.uint8, device="cuda")
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        for _ in range(2):
            sampler.sample_device(device[0].data_ptr(), hip_sampler.LOGITS_BF16 if dtype == "bf16" else hip_sampler.LOGITS_F32, rows, vocab, vocab,
                                  device[1].data_ptr(), device[2].data_ptr(), None, results.data_ptr(), hip_sampler.PASSES_FULL_ORDER,
                                  torch.cuda.current_stream().cuda_stream)
            gpu = results.cpu().numpy().view(hip_sampler.RESULT_DTYPE)
            parity_util.assert_results_match(gpu, cpu, dtype, "edges of parts")
            results.zero_()


@pytest.mark.parametrize("rows,vocab,top_ks", [(200, 8191, [300, 1000]), (96, 16411, [0, 300]), (40, 20011, [0])])
def test_calls_that_hold_each_other_s_places(rows, vocab, top_ks):
    """Three handles on three streams: workgroups of one call start when others of it have finished their rows, the soonest those
    that have no finite logit, and come to the same list of rows all the same.  Parts that hold places each other's rows need give their rows up;
    a call by itself then serves all that it served before."""
    print("[case] three streams, %d x %d, top_k %s" % (rows, vocab, top_ks), flush=True)
    calls = []
    for seed in range(3):
        rng = np.random.default_rng(rows + seed)
        logits = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
        logits[seed::7] = -np.inf
        params = hip_sampler.make_params(rows, 0.9, 0, 0.95, 0.0)
        params["top_k"] = rng.choice(top_ks, rows)
        uniforms = rng.random(rows, dtype=np.float32)
        device = [torch.from_numpy(x).cuda() for x in (logits, params.view(np.uint8), uniforms)]
        results = torch.zeros(8, rows * 16, dtype=torch.uint8, device="cuda")
        sampler = hip_sampler.HipSampler(rows, vocab, testing=True)
        sampler.binned_sums(True)
        calls.append((sampler, torch.cuda.Stream(), device, results, parity_util.run_oracle(logits, params, uniforms)))
    torch.cuda.synchronize()

    def last_served(call):
        top_k = call[2][1].cpu().numpy().view(hip_sampler.PARAMS_DTYPE)["top_k"]
        return int(call[0].binned_rows(rows)[top_k == 0].sum())

    def served(call):
        sampler, stream, device, results, _ = call
        sampler.sample_device(device[0].data_ptr(), hip_sampler.LOGITS_F32, rows, vocab, vocab, device[1].data_ptr(), device[2].data_ptr(), None,
                              results[0].data_ptr(), hip_sampler.PASSES_FULL_ORDER, stream.cuda_stream)
        torch.cuda.synchronize()
        return last_served(call)

    alone = [served(call) for call in calls]
    assert 0 not in top_ks or min(alone) > 0
    for i in range(8):
        for sampler, stream, device, results, _ in calls:
            sampler.sample_device(device[0].data_ptr(), hip_sampler.LOGITS_F32, rows, vocab, vocab, device[1].data_ptr(), device[2].data_ptr(), None,
                                  results[i].data_ptr(), hip_sampler.PASSES_FULL_ORDER, stream.cuda_stream)
    torch.cuda.synchronize()
    for sampler, _, _, results, cpu in calls:
        for i in range(8):
            gpu = results[i].cpu().numpy().view(hip_sampler.RESULT_DTYPE)
            parity_util.assert_results_match(gpu, cpu, "f32", "call %d beside others" % i)
    print("[served] alone %s, the last of the calls beside others %s" % (
        alone, [last_served(call) for call in calls]), flush=True)
    assert [served(call) for call in calls] == alone
    for sampler, *_ in calls:
        sampler.close()
