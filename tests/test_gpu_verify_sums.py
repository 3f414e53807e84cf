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
