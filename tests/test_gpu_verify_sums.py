"""Verification steps without a Top-K window (GPU): served from the rows' sums, with the residual as a dense vector in
chunks of 4,096 entries, at vocabularies around a chunk and for steps that accept everything, some or nothing."""
import numpy as np
import pytest

import test_gpu_speculative as speculative
from ncnn_moe_runtime_amd import hip_sampler

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("vocab,drafts", [(70, 1), (4095, 2), (4097, 5), (40961, 3), (151936, 5), (9000, 16)])
def test_steps_without_a_window_match_the_oracle(vocab, drafts, bf16):
    rng = np.random.default_rng(vocab + drafts)
    with hip_sampler.HipSampler(2 * drafts + 1, vocab) as sampler:
        for trial in range(6):
            spread = float(rng.choice([0.3, 2.0, 3.0]))
            options = dict(temperature=float(rng.choice([0.5, 1.0, 1.4])), top_p=float(rng.choice([0.5, 0.95, 0.999, 1.0])),
                           min_p=float(rng.choice([0.0, 0.0, 0.001])))
            target = (rng.standard_normal((drafts + 1, vocab)) * spread).astype(np.float32)
            noise = float(rng.choice([0.0, 0.1, 1.5]))
            draft = (target[:drafts] + noise * rng.standard_normal((drafts, vocab))).astype(np.float32)
            proposed = speculative._propose(rng, speculative.workloads.bf16_bits_to_float32(
                speculative.workloads.float32_to_bf16_bits(draft)) if bf16 else draft, options)
            if trial == 4:
                proposed[-1] = int(np.argmin(draft[-1]))  # hardly or not in the draft's distribution
            uniforms = rng.random(drafts + 1, dtype=np.float32)
            if trial == 5:
                uniforms[1:] = np.float32(1.0) - np.float32(2.0 ** -24)
            speculative._compare(sampler, target, draft, proposed, uniforms, "%d drafts over %d, trial %d" % (drafts, vocab, trial), bf16=bf16, **options)


@pytest.mark.parametrize("vocab,top_k,min_p", [(40961, 0, 0.02), (151936, 0, 0.001), (151936, 0, 2e-5), (40961, 30000, 0.02), (9000, 0, 1e-3)])
def test_steps_whose_min_p_cut_lies_behind_the_head(vocab, top_k, min_p):
    """The filtered distribution that a Min-P cut ends thousands of tokens down is known by the smallest term that it keeps: the
    step is not run a second time with exported lists."""
    rng = np.random.default_rng(vocab + top_k)
    drafts = 3
    with hip_sampler.HipSampler(2 * drafts + 1, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        for trial in range(4):
            options = dict(temperature=1.0, top_p=1.0 if trial % 2 else 0.9999, min_p=min_p, top_k=top_k)
            target = (rng.standard_normal((drafts + 1, vocab)) * 1.2).astype(np.float32)
            draft = (target[:drafts] + (0.1 if trial < 3 else 2.0) * rng.standard_normal((drafts, vocab))).astype(np.float32)
            proposed = speculative._propose(rng, draft, options)
            uniforms = rng.random(drafts + 1, dtype=np.float32)
            if trial >= 2:
                uniforms[1] = np.float32(1.0) - np.float32(2.0 ** -24)
            speculative._compare(sampler, target, draft, proposed, uniforms, "cut at %g over %d, trial %d" % (min_p, vocab, trial), **options)
            assert sampler.filtered_rows(2 * drafts + 1).tolist() == [1] * (2 * drafts + 1)
