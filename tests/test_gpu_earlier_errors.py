"""An error that an earlier, unrelated call left on the thread is no error of the calls behind it: they succeed, their results are right, and so are
those of the calls that follow."""
import contextlib

import numpy as np
import pytest

import oracle_lib
import parity_util
from ncnn_moe_runtime_amd import hip_router, hip_sampler

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

NO_SUCH_DEVICE = 1 << 20


def _leave_an_error(library):
    assert library.hipSetDevice(NO_SUCH_DEVICE) != 0


# (one launch whose records are watched, windows, no windows, and rows that the sort takes)
@pytest.mark.parametrize("top_k,binned", [(20, True), (300, True), (0, True), (0, False)])
def test_sample(top_k, binned):
    rows, vocab = 5, 20011
    rng = np.random.default_rng(top_k)
    params = hip_sampler.make_params(rows, 0.8, top_k, 0.9, 0.0)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(binned)
        for turn in range(3):
            print("[case] sample behind an error, top %d, turn %d" % (top_k, turn), flush=True)
            logits = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
            uniforms = rng.random(rows, dtype=np.float32)
            cpu = parity_util.run_oracle(logits, params, uniforms)
            sampler.upload_logits(logits)
            _leave_an_error(sampler._lib)
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "behind an error")
        _leave_an_error(sampler._lib)
        status, ids, probabilities, count = sampler.distribution(2, temperature=0.8, top_k=50, top_p=0.9)
        _, cpu_ids, cpu_probabilities = oracle_lib.oracle_distribution(logits[2], temperature=0.8, top_k=50, top_p=0.9)
        assert status == 0 and np.array_equal(ids, cpu_ids) and count == len(cpu_ids)
        np.testing.assert_allclose(probabilities, cpu_probabilities, rtol=parity_util.PROBABILITY_RTOL["f32"])


# (lists, the binned sums, and lists of whole rows)
@pytest.mark.parametrize("top_k,binned", [(50, True), (0, True), (0, False)])
def test_verification(top_k, binned):
    drafts, vocab = 2, 20011
    rows = 2 * drafts + 1
    rng = np.random.default_rng(top_k + 1)
    options = dict(temperature=0.9, top_k=top_k, top_p=0.95)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(binned)
        for turn in range(3):
            print("[case] verification behind an error, top %d, turn %d" % (top_k, turn), flush=True)
            target = (rng.standard_normal((drafts + 1, vocab)) * 2).astype(np.float32)
            draft = target[:drafts] + (rng.standard_normal((drafts, vocab)) * 0.5).astype(np.float32)
            proposed = [int(oracle_lib.oracle_sample(draft[i], 0.4, **options)["token_id"]) for i in range(drafts)]
            uniforms = rng.random(drafts + 1, dtype=np.float32)
            expected, expected_accepted = oracle_lib.oracle_speculative_verify(target, draft, proposed, uniforms, **options)
            sampler.upload_logits(np.concatenate([target, draft]))
            _leave_an_error(sampler._lib)
            verified, accepted = sampler.speculative_verify(proposed, uniforms, **options)
            assert verified.tobytes() == expected.tobytes() and accepted.tobytes() == expected_accepted.tobytes()


def test_device_entries():
    rows, vocab = 4, 20011
    rng = np.random.default_rng(3)
    params = hip_sampler.make_params(rows, 0.8, 20, 0.9, 0.0)
    logits = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
    uniforms = rng.random(rows, dtype=np.float32)
    cpu = parity_util.run_oracle(logits, params, uniforms)
    operands = [torch.from_numpy(x.view(np.uint8).copy()).cuda() for x in (logits, params, uniforms)]
    pointers = [x.data_ptr() for x in operands]
    results = torch.zeros(rows * 16, dtype=torch.uint8, device="cuda:0")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()

    def check(context):
        stream.synchronize()
        parity_util.assert_results_match(results.cpu().numpy().view(hip_sampler.RESULT_DTYPE).reshape(rows), cpu, "f32", context)
        results.zero_()
        torch.cuda.synchronize()

    with hip_sampler.HipSampler(rows, vocab) as sampler:
        for turn in range(2):
            print("[case] device entries behind an error, turn %d" % turn, flush=True)
            _leave_an_error(sampler._lib)
            sampler.sample_device(pointers[0], hip_sampler.LOGITS_F32, rows, vocab, vocab, pointers[1], pointers[2], None, results.data_ptr(), 0, stream.cuda_stream)
            check("sample_device")
            _leave_an_error(sampler._lib)
            assert hip_sampler.sample_device_static(0, pointers[0], hip_sampler.LOGITS_F32, rows, vocab, vocab, pointers[1], pointers[2], None, results.data_ptr(), stream.cuda_stream) == 0
            check("sample_device_static")


@pytest.mark.parametrize("tokens", [40, 600])
def test_router(tokens):
    experts, top_k = 64, 6
    rng = np.random.default_rng(tokens)
    with contextlib.closing(hip_router.HipRouter(tokens, experts, top_k)) as router:
        for turn in range(2):
            print("[case] router behind an error, %d tokens, turn %d" % (tokens, turn), flush=True)
            logits = rng.standard_normal((tokens, experts)).astype(np.float32)
            cpu_status, cpu_offsets, cpu_routes = oracle_lib.oracle_router_dispatch(logits, top_k)
            _leave_an_error(hip_router.load_library())
            status, offsets, routes = router.dispatch(logits, top_k)
            assert status == cpu_status == 0 and np.array_equal(offsets, cpu_offsets)
            for field in ("token_index", "rank"):
                assert np.array_equal(routes[field], cpu_routes[field]), field
            assert np.array_equal(routes["weight"].view(np.uint32), cpu_routes["weight"].view(np.uint32))
