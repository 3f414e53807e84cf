"""ncnn_moe_hip_sampler_sample_device through the C ABI with every operand in device memory (torch only
allocates the buffers and owns the stream): the entry the decode step calls.  Checks the three
passes (batch-shaped select, wide select, full order), the may_need_full_order contract and that the
call does not need the handle's own logits buffer."""
import numpy as np
import pytest

import parity_util
from ncnn_moe_runtime_amd import hip_sampler

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _device(array):
    return torch.from_numpy(np.ascontiguousarray(array).view(np.uint8).reshape(-1)).to("cuda:0")


def _run(sampler, logits, params, uniforms, may_need_full_order, stream):
    rows, vocab = logits.shape
    dtype = hip_sampler.LOGITS_F32 if logits.dtype == np.float32 else hip_sampler.LOGITS_BF16
    d_logits, d_params, d_uniforms = _device(logits), _device(params), _device(uniforms)
    d_results = torch.zeros(rows * 16, dtype=torch.uint8, device="cuda:0")
    torch.cuda.synchronize()
    sampler.sample_device(d_logits.data_ptr(), dtype, rows, vocab, vocab, d_params.data_ptr(), d_uniforms.data_ptr(),
                          None, d_results.data_ptr(), may_need_full_order, stream.cuda_stream)
    stream.synchronize()
    return d_results.cpu().numpy().view(hip_sampler.RESULT_DTYPE).reshape(rows)


@pytest.mark.parametrize("rows", [24, 300])
def test_three_passes_on_a_caller_stream(rows):
    print("[case] sample_device, %d rows, mixed windows" % rows, flush=True)
    rng = np.random.default_rng(rows)
    vocab = 50021
    logits = (rng.standard_normal((rows, vocab)) * 2.5).astype(np.float32)
    params = hip_sampler.make_params(rows, 0.8, 0, 0.92, 0.0)
    params["top_k"] = np.array([(1, 20, 64, 65, 700, 1024, 1025, 0)[i % 8] for i in range(rows)], dtype=np.uint32)
    params["temperature"][::11] = 0.0
    uniforms = rng.random(rows).astype(np.float32)
    cpu = parity_util.run_oracle(logits, params, uniforms)
    stream = torch.cuda.Stream(device="cuda:0")
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        full = _run(sampler, logits, params, uniforms, True, stream)
        parity_util.assert_results_match(full, cpu, "f32", "sample_device, all passes")
        served_by_select = (params["temperature"] == 0.0) | ((params["top_k"] >= 1) & (params["top_k"] <= 1024))
        assert ((full["flags"][served_by_select] & hip_sampler.FLAG_GENERAL_PATH) == 0).all()
        # one kernel only: rows that need a later pass say so, the others are final
        first = _run(sampler, logits, params, uniforms, False, stream)
        narrow = (params["temperature"] == 0.0) | ((params["top_k"] >= 1) & (params["top_k"] <= 64))
        assert (first["status"][~narrow] == hip_sampler.ROW_NEEDS_FULL_ORDER).all()
        assert (first["token_id"][~narrow] == -1).all()
        parity_util.assert_results_match(first[narrow], cpu[narrow], "f32", "sample_device, select pass only")
        # and a second call with every pass finishes them
        again = _run(sampler, logits, params, uniforms, True, stream)
        parity_util.assert_results_match(again, cpu, "f32", "sample_device, repeated")


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_later_passes_side_by_side(dtype):
    """Rows with wide windows and rows without a window in one batch: the wide select on the handle's
    second stream beside the full-order kernels (flag NCNN_MOE_PASSES_SIDE_BY_SIDE, and sample() by
    itself from 32 rows of each kind), with tie-heavy rows that the wide select, and the first select for a
    window of 20, hand on to the full-order kernels behind the join.  Same results as one pass after the
    other, and as the oracle."""
    print("[case] later passes side by side, %s" % dtype, flush=True)
    from ncnn_moe_runtime_amd import workloads
    rng = np.random.default_rng(77)
    rows, vocab = 120, 30011
    logits = (rng.standard_normal((rows, vocab)) * 2.0).astype(np.float32)
    logits[5::12] = np.round(logits[5::12])  # a few thousand equal logits around every cut
    logits[2::12] = np.round(logits[2::12] / 2.0) * 2.0  # (top_k 20: hundreds of equal logits at the cut)
    params = hip_sampler.make_params(rows, 0.9, 0, 0.9, 0.0)
    params["top_k"] = np.array([(700, 0, 20, 300, 2000, 1024)[i % 6] for i in range(rows)], dtype=np.uint32)
    params["temperature"][::17] = 0.0
    uniforms = rng.random(rows).astype(np.float32)
    data = workloads.float32_to_bf16_bits(logits) if dtype == "bf16" else logits
    cpu = parity_util.run_oracle(data, params, uniforms)
    stream = torch.cuda.Stream(device="cuda:0")
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        in_turn = _run(sampler, data, params, uniforms, hip_sampler.PASSES_FULL_ORDER, stream)
        beside = _run(sampler, data, params, uniforms, hip_sampler.PASSES_FULL_ORDER | hip_sampler.PASSES_SIDE_BY_SIDE, stream)
        # (a row that the first select hands on is served by the wide select when the passes run in turn and by
        # the full-order kernels behind the join when they run side by side: the same result, and the flag
        # that names the path differs)
        handed_on = np.zeros(rows, dtype=bool)
        handed_on[2::12] = params["temperature"][2::12] != 0.0
        assert in_turn[~handed_on].tobytes() == beside[~handed_on].tobytes()
        assert ((beside["flags"] ^ in_turn["flags"])[handed_on] == hip_sampler.FLAG_GENERAL_PATH).all()
        for field in beside.dtype.names:
            if field != "flags":
                assert in_turn[field].tobytes() == beside[field].tobytes(), field
        parity_util.assert_results_match(beside, cpu, dtype, "side by side, device entry")
        for _ in range(3):  # the second stream forks and joins again on every call
            again = _run(sampler, data, params, uniforms, hip_sampler.PASSES_FULL_ORDER | hip_sampler.PASSES_SIDE_BY_SIDE, stream)
            assert again.tobytes() == beside.tobytes()
        sampler.upload_logits(data)
        host = sampler.sample(params, uniforms)
        parity_util.assert_results_match(host, cpu, dtype, "side by side, host entry")


def test_bf16_strided_rows_on_the_default_stream():
    print("[case] sample_device, bf16, stride wider than the vocabulary", flush=True)
    from ncnn_moe_runtime_amd import workloads
    rng = np.random.default_rng(5)
    rows, vocab, stride = 70, 40001, 40008
    values = (rng.standard_normal((rows, stride)) * 2).astype(np.float32)
    bits = workloads.float32_to_bf16_bits(values)
    bits[:, vocab:] = workloads.float32_to_bf16_bits(np.full((rows, stride - vocab), 60.0, dtype=np.float32))  # never read
    params = hip_sampler.make_params(rows, 0.7, 40, 0.9, 0.01)
    uniforms = rng.random(rows).astype(np.float32)
    cpu = parity_util.run_oracle(np.ascontiguousarray(bits[:, :vocab]), params, uniforms)
    d_logits, d_params, d_uniforms = _device(bits), _device(params), _device(uniforms)
    d_results = torch.zeros(rows * 16, dtype=torch.uint8, device="cuda:0")
    torch.cuda.synchronize()
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.sample_device(d_logits.data_ptr(), hip_sampler.LOGITS_BF16, rows, vocab, stride, d_params.data_ptr(),
                              d_uniforms.data_ptr(), None, d_results.data_ptr(), False, None)
        torch.cuda.synchronize()
    gpu = d_results.cpu().numpy().view(hip_sampler.RESULT_DTYPE).reshape(rows)
    parity_util.assert_results_match(gpu, cpu, "bf16", "sample_device, bf16 strided")


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_no_wide_windows_flag(dtype):
    """NCNN_MOE_PASSES_NO_WIDE_WINDOWS leaves out the select kernel for 64 < top_k <= 1024.  With no such row
    the results are those of the full set of passes; a row that has such a window after all (the caller's
    promise broken) is served by the full-order kernels, with the same result."""
    print("[case] sample_device without the wide select, %s" % dtype, flush=True)
    from ncnn_moe_runtime_amd import workloads
    rng = np.random.default_rng(404)
    rows, vocab = 96, 40013
    logits = (rng.standard_normal((rows, vocab)) * 2.0).astype(np.float32)
    data = workloads.float32_to_bf16_bits(logits) if dtype == "bf16" else logits
    params = hip_sampler.make_params(rows, 0.9, 0, 0.9, 0.0)
    params["top_k"] = np.array([(0, 20, 5000, 1, 64, 0)[i % 6] for i in range(rows)], dtype=np.uint32)
    uniforms = rng.random(rows).astype(np.float32)
    stream = torch.cuda.Stream(device="cuda:0")
    flags = hip_sampler.PASSES_FULL_ORDER | hip_sampler.PASSES_NO_WIDE_WINDOWS
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        cpu = parity_util.run_oracle(data, params, uniforms)
        every_pass = _run(sampler, data, params, uniforms, hip_sampler.PASSES_FULL_ORDER, stream)
        without = _run(sampler, data, params, uniforms, flags, stream)
        assert every_pass.tobytes() == without.tobytes()
        parity_util.assert_results_match(without, cpu, dtype, "no wide windows")
        params["top_k"][3::6] = 700   # wide windows after all
        cpu = parity_util.run_oracle(data, params, uniforms)
        broken_promise = _run(sampler, data, params, uniforms, flags | hip_sampler.PASSES_SIDE_BY_SIDE, stream)
        parity_util.assert_results_match(broken_promise, cpu, dtype, "wide windows without the wide select")
        assert (broken_promise["flags"][3::6] & hip_sampler.FLAG_GENERAL_PATH != 0).all()


def test_rejected_rows_side_by_side():
    """Rows without a finite logit, or with +inf, among the rows that the first select marks as pending on the second stream
    while their sums begin on the caller's: rejected in every call, none left pending."""
    print("[case] rejected rows side by side", flush=True)
    rng = np.random.default_rng(78)
    rows, vocab = 192, 20011
    logits = (rng.standard_normal((rows, vocab)) * 2.0).astype(np.float32)
    logits[0::6] = -np.inf
    logits[1::6, vocab - 1] = np.inf
    logits[2::12] = np.nan
    params = hip_sampler.make_params(rows, 0.9, 0, 0.9, 0.0)
    params["top_k"] = np.array([(0, 0, 0, 700, 300, 0, 0)[i % 7] for i in range(rows)], dtype=np.uint32)
    uniforms = rng.random(rows).astype(np.float32)
    cpu = parity_util.run_oracle(logits, params, uniforms)
    stream = torch.cuda.Stream(device="cuda:0")
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(logits)
        for _ in range(4):
            beside = _run(sampler, logits, params, uniforms, hip_sampler.PASSES_FULL_ORDER | hip_sampler.PASSES_SIDE_BY_SIDE, stream)
            parity_util.assert_results_match(beside, cpu, "f32", "rejected rows, device entry")
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "rejected rows, host entry")


@pytest.mark.parametrize("rows", [1, 63, 65, 1023, 1024, 1025, 2050])
def test_rows_listed_by_the_first_launch_or_by_one_of_their_own(rows):
    """Up to 1,024 rows the launches that want a list of rows make it themselves: of each kind, alone, together and side by side."""
    rng = np.random.default_rng(rows)
    vocab = 1211
    print("[case] %d rows listed" % rows, flush=True)
    logits = (rng.standard_normal((rows, vocab)) * 2.0).astype(np.float32)
    uniforms = rng.random(rows).astype(np.float32)
    stream = torch.cuda.Stream(device="cuda:0")
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        for kinds in ((20, 0, 200, 1000), (0,), (200,), (20,)):
            params = hip_sampler.make_params(rows, 0.9, 0, 0.93, 0.0)
            params["top_k"] = rng.choice(np.array(kinds, dtype=np.uint32), rows)
            params["temperature"][::9] = 0.0
            cpu = parity_util.run_oracle(logits, params, uniforms)
            flags = [hip_sampler.PASSES_FULL_ORDER, hip_sampler.PASSES_FULL_ORDER | hip_sampler.PASSES_SIDE_BY_SIDE]
            if 200 not in kinds:
                flags.append(hip_sampler.PASSES_FULL_ORDER | hip_sampler.PASSES_NO_WIDE_WINDOWS)
            for passes in flags:
                gpu = _run(sampler, logits, params, uniforms, passes, stream)
                parity_util.assert_results_match(gpu, cpu, "f32", "%d rows of %s, passes %d" % (rows, kinds, passes))


@pytest.mark.parametrize("rows,vocab,windows,sums", [(320, 262147, 256, 36), (320, 262147, 256, 37), (320, 262143, 256, 36), (257, 262147, 256, 0), (1100, 65537, 1024, 40)])
def test_windows_that_go_ahead_of_the_sums(rows, vocab, windows, sums):
    """Side by side, windows of 2^26 logits and more and of seven rows and more for each row without one start before the sums'
    passes have ended: on both sides of both limits, with the rows listed in place and by a launch, eager and captured, the rows'
    results are those of the passes one behind the other, and the oracle's."""
    print("[case] windows ahead, %d x %d, %d windows, %d sums" % (rows, vocab, windows, sums), flush=True)
    rng = np.random.default_rng(windows + sums)
    generator = torch.Generator(device="cuda:0").manual_seed(vocab)
    d_logits = torch.randn(rows, vocab, device="cuda:0", generator=generator).mul_(2.0)
    params = hip_sampler.make_params(rows, 0.9, 20, 0.93, 0.0)
    kinds = rng.permutation(rows)
    params["top_k"][kinds[:windows]] = rng.choice(np.array([65, 300, 1024], dtype=np.uint32), windows)
    params["top_k"][kinds[windows:windows + sums]] = 0
    uniforms = rng.random(rows, dtype=np.float32)
    d_params, d_uniforms = _device(params.view(np.uint8)), _device(uniforms)
    d_results = torch.zeros(rows * 16, dtype=torch.uint8, device="cuda:0")
    stream = torch.cuda.Stream(device="cuda:0")
    torch.cuda.synchronize()
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        def enqueue(passes):
            sampler.sample_device(d_logits.data_ptr(), hip_sampler.LOGITS_F32, rows, vocab, vocab, d_params.data_ptr(), d_uniforms.data_ptr(),
                                  None, d_results.data_ptr(), passes, stream.cuda_stream)

        def results():
            torch.cuda.synchronize()
            out = d_results.cpu().numpy().view(hip_sampler.RESULT_DTYPE).reshape(rows)
            d_results.zero_()
            torch.cuda.synchronize()
            return out

        enqueue(hip_sampler.PASSES_FULL_ORDER)
        in_turn = results()
        beside_flags = hip_sampler.PASSES_FULL_ORDER | hip_sampler.PASSES_SIDE_BY_SIDE
        for _ in range(2):
            enqueue(beside_flags)
            assert results().tobytes() == in_turn.tobytes()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            enqueue(beside_flags)
        for _ in range(3):
            graph.replay()
            assert results().tobytes() == in_turn.tobytes()
    checked = np.concatenate([kinds[:8], kinds[windows:windows + min(sums, 8)], kinds[-4:]])
    cpu = parity_util.run_oracle(d_logits[torch.from_numpy(checked).to("cuda:0")].cpu().numpy(), params[checked], uniforms[checked])
    parity_util.assert_results_match(in_turn[checked], cpu, "f32", "windows ahead")
