"""Rows that the first select leaves, served by the window kernels and by sums over unordered bins of terms (GPU): the
oracle's results, on rows where the sums cross many binades, end inside the sorted head or far behind it, meet terms half way between two sums,
ties, cuts and windows, at the sizes where the parts and bins of a row begin and end."""
import numpy as np
import pytest

import parity_util
import test_gpu_speculative as speculative
from ncnn_moe_runtime_amd import hip_sampler, workloads

pytestmark = pytest.mark.gpu


def _batch(rng, rows, vocab, top_k):
    logits = (rng.standard_normal((rows, vocab)) * rng.uniform(0.3, 3.0, (rows, 1))).astype(np.float32)
    kinds = np.arange(rows) % 8
    logits[kinds == 1] = np.round(logits[kinds == 1] * 16) / 16          # a few hundred values: large bins of equal terms
    logits[kinds == 2, ::97] += np.float32(9.0)                           # a peaked row
    logits[kinds == 3, vocab // 3:] = -np.inf                             # a masked vocabulary
    logits[kinds == 4] = logits[kinds == 4] * np.float32(0.01) + np.float32(40.0)  # narrow: every term in one binade
    logits[kinds == 5, vocab // 2] = np.nan
    params = hip_sampler.make_params(rows, 1.0, 0, 1.0, 0.0)
    params["temperature"] = rng.choice(np.array([0.2, 0.7, 1.0, 1.3, 2.5], dtype=np.float32), rows)
    params["top_k"] = rng.choice(np.array(top_k, dtype=np.uint32), rows)
    params["top_p"] = rng.choice(np.array([0.3, 0.8, 0.95, 0.999, 1.0], dtype=np.float32), rows)
    params["min_p"] = rng.choice(np.array([0.0, 0.0, 1e-4, 0.02], dtype=np.float32), rows)
    return logits, params, rng.random(rows, dtype=np.float32)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("rows,vocab", [(1, 151936), (3, 2047), (9, 8193), (8, 100003), (40, 32771), (130, 16411), (520, 2049)])
def test_binned_sums_match_the_oracle(dtype, rows, vocab):
    rng = np.random.default_rng(rows * 1000003 + vocab)
    # (bf16 rows without a window have a kernel of their own)
    top_k = [0, 0, 65, 1000, 1025, 5000, vocab - 1] if dtype == "f32" else [65, 200, 700, 1024]
    print("[case] binned sums, %d x %d %s" % (rows, vocab, dtype), flush=True)
    logits, params, uniforms = _batch(rng, rows, vocab, top_k)
    data = workloads.float32_to_bf16_bits(logits) if dtype == "bf16" else logits
    cpu = parity_util.run_oracle(data, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.upload_logits(data)
        sorted_way = sampler.sample(params, uniforms)
        sampler.binned_sums(True)
        gpu = sampler.sample(params, uniforms)
        windows = (params["top_k"] > 0) & (params["top_k"] <= 1024) | (vocab <= 1024)
        general = (gpu["flags"] & hip_sampler.FLAG_GENERAL_PATH) != 0
        served = np.where(windows, ~general, sampler.binned_rows(rows) == 1)
        again = sampler.sample(params, uniforms)
    parity_util.assert_results_match(gpu, cpu, dtype, "binned sums")
    for field in ("token_id", "probability", "kept_count", "status", "draw_consumed"):
        assert gpu[field].tobytes() == sorted_way[field].tobytes(), field
    assert gpu.tobytes() == again.tobytes()
    # what is left to the sort is the exception: thousands of equal terms, and draws that no partial sum exceeds
    assert served.sum() >= rows - 1 - rows // 5, (served, rows)


def test_draws_and_cuts_at_the_ends():
    """Draws at the ends of [0, 1), Min-P cuts at and behind the last bin, a Top-P that the first element meets."""
    rng = np.random.default_rng(99)
    rows, vocab = 24, 50021
    logits, params, uniforms = _batch(rng, rows, vocab, [0, 0, 3000])
    uniforms[0::3] = 0.0
    uniforms[1::3] = np.float32(1.0) - np.float32(2.0 ** -24)
    params["min_p"][2::4] = np.float32(1e-7)
    params["min_p"][3::4] = np.float32(1e-30)
    params["top_p"][::5] = np.float32(1e-6)
    params["min_p"][::7] = 1.0
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.upload_logits(logits)
        gpu = sampler.sample(params, uniforms)
    parity_util.assert_results_match(gpu, cpu, "f32", "ends")


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("rows,vocab", [(12, 2049), (12, 16411), (300, 4099)])
def test_quotients_and_finite_counts_at_the_ends_of_their_ranges(dtype, rows, vocab):
    """Temperatures on both sides of those whose quotients are made with corrections, a maximum next to zero among tiny logits, and rows with NaN,
    -inf and the largest numbers at their ends and inside, in one launch and in four, fp32 rows in windows and without one, bf16 rows in windows (the limits of
    logits and maxima, and bf16 rows without a window: the tests behind this one)."""
    rng = np.random.default_rng(rows + vocab)
    print("[case] ends of quotients, %d x %d %s" % (rows, vocab, dtype), flush=True)
    logits = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
    params = hip_sampler.make_params(rows, 1.0, 0, 0.95, 0.0)
    scales = 2.0 ** np.array([0, 0, -19.5, -20.5, 19.5, 20.5, -90, 59, 61, 0, 0, 0], dtype=np.float64)
    kinds = np.arange(rows) % 12
    params["temperature"] = np.clip(scales, 2.0 ** -21, 2.0 ** 21)[kinds].astype(np.float32)
    logits = (logits * scales[kinds][:, None]).astype(np.float32)
    logits[kinds == 1] -= logits[kinds == 1].max(axis=1, keepdims=True)      # a maximum of zero
    logits[kinds == 9] = logits[kinds == 9] - logits[kinds == 9].max(axis=1, keepdims=True) + np.float32(2.0 ** -21)
    logits[kinds == 9, ::5] = np.float32(-1e-39)
    logits[kinds == 10, ::3] = -np.inf
    for at in (0, vocab // 2, vocab - 1):
        logits[kinds == 10, at] = np.nan
    logits[kinds == 11, 0] = logits[kinds == 11, vocab - 1] = np.float32(-3.0e38)
    if dtype == "bf16":
        params["top_k"] = 100
    else:
        params["top_k"][rows // 2::2] = 100
    uniforms = rng.random(rows, dtype=np.float32)
    data = workloads.float32_to_bf16_bits(logits) if dtype == "bf16" else logits
    cpu = parity_util.run_oracle(data, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.upload_logits(data)
        gpu = sampler.sample(params, uniforms)
    parity_util.assert_results_match(gpu, cpu, dtype, "ends of quotients")


# Terms are made with corrected quotients for temperatures of 2^-20 to 2^20 where no logit is beyond 2^60 and the maximum is 2^-20 at least: a row for each
# side of each limit, its logits ordinary ones but for those that the limit is about.  `below` and `above`: the neighbours in the row's type.
LIMIT_KINDS = ["ordinary", "logit 2^60", "logit above 2^60", "maximum 2^-20", "maximum below 2^-20", "maximum above 2^-20", "ends"]


def _limit_row(rng, kind, vocab, temperature, spread, below, above):
    row = (rng.standard_normal(vocab) * spread * temperature).astype(np.float32)
    if kind.startswith("logit"):
        limit = np.float32(2.0 ** 60)
        row[vocab // 3] = -(limit if kind == "logit 2^60" else above(limit))
    elif kind.startswith("maximum"):
        # (the maximum is the largest logit by the temperature, which is a power of two in these rows)
        limit = np.float32(2.0 ** -20) * np.float32(temperature)
        row = -np.abs(row) - np.float32(temperature) * np.float32(0.01)
        row[::997] = np.float32(-1e-39)  # (some hundred: rows of thousands of equal terms, which these all are to the maximum, are sorted)
        row[1::997] = np.float32(2.0 ** -75)
        row[vocab // 3] = below(limit) if "below" in kind else above(limit) if "above" in kind else limit
    elif kind == "ends":
        row[1::7] = -np.inf
        row[0] = row[vocab // 2] = row[-1] = np.nan
        row[2] = row[-2] = np.float32(-2.0 ** 60)
    return row


def _float_below(x):
    return np.nextafter(np.float32(x), np.float32(0))


def _float_above(x):
    return np.nextafter(np.float32(x), np.float32(np.inf))


# (one launch, and four)
@pytest.mark.parametrize("rows,vocab", [(49, 4099), (5, 16411), (294, 2053)])
def test_quotients_at_the_limits_of_logits_and_maxima(rows, vocab):
    rng = np.random.default_rng(rows + vocab)
    print("[case] limits of quotients, %d x %d" % (rows, vocab), flush=True)
    temperatures = [1.0, 0.7, 1.3 * 2.0 ** 19, 2.0 ** 20, _float_above(2.0 ** 20), 2.0 ** -20, _float_below(2.0 ** -20)]
    logits = np.empty((rows, vocab), dtype=np.float32)
    params = hip_sampler.make_params(rows, 1.0, 0, 0.999, 0.0)
    for row in range(rows):
        kind = LIMIT_KINDS[row % 7]
        temperature = np.float32(2.0 ** (row // 7 % 3 * 9) if kind.startswith("maximum") else temperatures[row // 7 % 7])
        params["temperature"][row] = temperature
        params["top_p"][row] = (0.9, 0.999, 1.0)[row // 49 % 3]
        logits[row] = _limit_row(rng, kind, vocab, temperature, 2.0, _float_below, _float_above)
    uniforms = rng.random(rows, dtype=np.float32)
    cpu = parity_util.run_oracle(logits, params, uniforms)
    assert (cpu["kept_count"] > 100).all()  # (the rows' sums are of many terms)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.upload_logits(logits)
        gpu = sampler.sample(params, uniforms)
        served = sampler.binned_rows(rows)
    parity_util.assert_results_match(gpu, cpu, "f32", "limits of quotients")
    assert served.sum() >= rows - 1 - rows // 5, (served, rows)


# bf16 rows without a window come to these kernels by the verification.  (One launch, and four: parts of more than 20,000 logits.)
@pytest.mark.parametrize("drafts,vocab", [(3, 4099), (1, 320103)])
@pytest.mark.parametrize("temperature", [1.0, 0.7, 1.3 * 2.0 ** 19, 2.0 ** 20, 2.0 ** 21, 2.0 ** -20, 2.0 ** -21])
def test_quotients_of_bf16_rows_at_their_limits(drafts, vocab, temperature):
    rng = np.random.default_rng(drafts + vocab)
    options = dict(temperature=temperature, top_p=0.999)
    step = 2.0 ** -7

    def below(x):
        return np.float32(x) * np.float32(1 - step / 2)

    def above(x):
        return np.float32(x) * np.float32(1 + step)

    def rounded(x):
        return workloads.bf16_bits_to_float32(workloads.float32_to_bf16_bits(x))

    kinds = LIMIT_KINDS if np.log2(temperature) % 1 == 0 else [kind for kind in LIMIT_KINDS if not kind.startswith("maximum")]
    with hip_sampler.HipSampler(2 * drafts + 1, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        served = 0
        for kind in kinds:
            print("[case] limits of bf16 quotients, %d drafts over %d, temperature %g, %s" % (drafts, vocab, temperature, kind), flush=True)
            target = rounded(np.stack([_limit_row(rng, kind, vocab, temperature, 2.0, below, above) for _ in range(drafts + 1)]))
            noise = 1 + (0.1 * rng.standard_normal((drafts, vocab))).astype(np.float32)
            draft = target[:drafts] * np.where(np.abs(target[:drafts]) > 2.0 ** 50, 1, noise).astype(np.float32)
            if kind.startswith("maximum"):
                draft[:, vocab // 3] = target[:drafts, vocab // 3]
            draft = rounded(draft)
            proposed = speculative._propose(rng, draft, options)
            uniforms = rng.random(drafts + 1, dtype=np.float32)
            speculative._compare(sampler, target, draft, proposed, uniforms, kind, bf16=True, **options)
            served += int(sampler.filtered_rows(2 * drafts + 1).sum())
    # (rows of hundreds of thousands of bf16 logits hold so many equal ones that some are left to the sort)
    assert served >= (2 * drafts + 1) * len(kinds) // 2, served


# Both sides of what decides whether the sums are one launch: elements a part (16 parts of 20,000 logits, and 6 of 80,000 where the call has
# windows), and as many rows as compute units.
@pytest.mark.parametrize("rows,vocab,windows", [(16, 65537, 0), (17, 65537, 0), (3, 320015, 0), (3, 320016, 0), (256, 4099, 0), (257, 4099, 0),
                                                (40, 480005, 3), (40, 480006, 3), (256, 4099, 20), (257, 4099, 20)])
@pytest.mark.parametrize("apart", [False, True])
def test_sums_of_one_launch_and_of_four(rows, vocab, windows, apart):
    """Many ties half way between two sums, which the walks fetch; with parts that hand over inside an XCD, and as if between them."""
    rng = np.random.default_rng(rows)
    print("[case] one launch and four, %d x %d, %d windows, apart %d" % (rows, vocab, windows, apart), flush=True)
    logits, params, uniforms = _batch(rng, rows, vocab, [0, 0, 5000])
    logits[::2] = rng.integers(-400, 400, (len(logits[::2]), vocab)).astype(np.float32) / 128
    params["temperature"][::2] = 1.0
    params["top_k"][rows - windows:] = 300
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.parts_apart(apart)
        sampler.upload_logits(logits)
        gpu = sampler.sample(params, uniforms)
        served = sampler.binned_rows(rows)[params["top_k"] != 300].sum()
        again = sampler.sample(params, uniforms)
    parity_util.assert_results_match(gpu, cpu, "f32", "one launch and four")
    assert gpu.tobytes() == again.tobytes()
    assert served > 0


@pytest.mark.parametrize("rows,vocab", [(8, 151936), (16, 40009), (40, 20011)])
def test_rows_whose_parts_do_not_wait_for_each_other(rows, vocab):
    """A part that finds the others missing gives its row up: the row is sorted, and the launches behind find everything as a
    finished row leaves it."""
    rng = np.random.default_rng(rows)
    print("[case] parts that do not wait, %d x %d" % (rows, vocab), flush=True)
    logits, params, uniforms = _batch(rng, rows, vocab, [0, 0, 5000])
    params["top_p"] = 1.0
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.upload_logits(logits)
        first = sampler.sample(params, uniforms)
        served = sampler.binned_rows(rows).sum()
        sampler.most_looks(0)
        for _ in range(3):
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "parts that do not wait")
        assert sampler.binned_rows(rows).sum() < served
        sampler.most_looks(40000)
        again = sampler.sample(params, uniforms)
        assert sampler.binned_rows(rows).sum() == served
    parity_util.assert_results_match(first, cpu, "f32", "parts that wait")
    assert first.tobytes() == again.tobytes()


@pytest.mark.parametrize("rows,vocab,top_ks", [(40, 151936, [0]), (300, 4099, [0]), (80, 33001, [0, 300])])
def test_rows_of_four_launches_whose_parts_do_not_wait_for_each_other(rows, vocab, top_ks):
    """The same where the walks are a launch of their own: six parts a row that meet first behind the first walk, one part a row, which
    meets nobody, and twelve beside the windows and the select."""
    rng = np.random.default_rng(rows + vocab)
    print("[case] four launches, parts that do not wait, %d x %d" % (rows, vocab), flush=True)
    logits, params, uniforms = _batch(rng, rows, vocab, [0])
    params["top_k"] = np.resize(np.array(top_ks, dtype=np.uint32), rows)
    params["top_p"] = 1.0
    sums = params["top_k"] == 0
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.upload_logits(logits)
        first = sampler.sample(params, uniforms)
        served = sampler.binned_rows(rows)[sums]
        sampler.most_looks(0)
        for _ in range(3):
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "parts that do not wait")
        given_up = served.sum() - sampler.binned_rows(rows)[sums].sum()
        assert given_up == 0 if rows == 300 else given_up > 0
        sampler.most_looks(40000)
        again = sampler.sample(params, uniforms)
        assert np.array_equal(sampler.binned_rows(rows)[sums], served)
    parity_util.assert_results_match(first, cpu, "f32", "parts that wait")
    assert first.tobytes() == again.tobytes()


@pytest.mark.parametrize("rows,vocab", [(1, 151936), (8, 151936), (40, 20011), (40, 151936), (130, 16411)])
def test_parts_that_hand_over_between_xcds(rows, vocab):
    """All that parts hand to each other in the launches of the sums, stored with agent scope, as where they are on several XCDs: the same
    results, from the sums."""
    rng = np.random.default_rng(rows * 7 + vocab)
    print("[case] parts apart, %d x %d" % (rows, vocab), flush=True)
    logits, params, uniforms = _batch(rng, rows, vocab, [0, 0, 5000])
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.upload_logits(logits)
        near = sampler.sample(params, uniforms)
        served = sampler.binned_rows(rows)
        sampler.parts_apart(True)
        for _ in range(3):
            apart = sampler.sample(params, uniforms)
            assert apart.tobytes() == near.tobytes()
            assert np.array_equal(sampler.binned_rows(rows), served)
    parity_util.assert_results_match(near, cpu, "f32", "parts apart")


@pytest.mark.parametrize("rows,vocab", [(8, 151936), (40, 151936), (5, 20011)])
def test_rows_cut_as_on_smaller_devices(rows, vocab):
    """Rows of eight parts, four and one, as on a device of 64 compute units, 32 and 8: the same results, from the sums."""
    rng = np.random.default_rng(rows + vocab)
    print("[case] smaller devices, %d x %d" % (rows, vocab), flush=True)
    logits, params, uniforms = _batch(rng, rows, vocab, [0, 0, 5000])
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.upload_logits(logits)
        first = sampler.sample(params, uniforms)
        served = sampler.binned_rows(rows).sum()
        for compute_units in (64, 32, 8):
            sampler.compute_units(compute_units)
            gpu = sampler.sample(params, uniforms)
            assert gpu.tobytes() == first.tobytes(), "as on %d compute units" % compute_units
            assert sampler.binned_rows(rows).sum() == served
        with pytest.raises(hip_sampler.SamplerError):
            sampler.compute_units(64)
    parity_util.assert_results_match(first, cpu, "f32", "all parts")


def _bf16_values(row):
    return workloads.bf16_bits_to_float32(workloads.float32_to_bf16_bits(row))


# (scale of the normal logits, what they are rounded to, Top-P, seeds): rows on which the sums foreseen from the bins are off
# by 1e-4 and more where the Top-P sum ends
FORESEEN_ENDS = [
    (2.5, "bf16", 0.98, (20,)),
    (2.5, "", 0.9999, (0, 17, 19, 21, 28)),
    (2.0, "eighths", 0.999, (0, 3, 9, 11)),
    (2.0, "eighths", 1.0, (3, 6, 20, 22)),
]


@pytest.mark.parametrize("scale,rounded,top_p,seeds", FORESEEN_ENDS)
def test_the_exact_sum_decides_where_the_top_p_sum_ends(scale, rounded, top_p, seeds):
    """A sum that the bins' masses foresee as ended goes on as long as the exact one has not reached its bound."""
    vocab = 151936
    logits = np.stack([(np.random.default_rng(seed).standard_normal(vocab) * scale).astype(np.float32) for seed in seeds])
    if rounded == "bf16":
        logits = _bf16_values(logits)
    elif rounded == "eighths":
        logits = np.round(logits * 8) / 8
    logits = np.ascontiguousarray(np.repeat(logits, 3, axis=0), dtype=np.float32)
    rows = len(logits)
    print("[case] foreseen ends, %g %s top_p %g" % (scale, rounded, top_p), flush=True)
    params = hip_sampler.make_params(rows, 1.0, 0, top_p, 0.0)
    uniforms = np.tile(np.array([0.25, 0.9, 1.0 - 2.0 ** -24], dtype=np.float32), len(seeds))
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(logits)
        gpu = sampler.sample(params, uniforms)
    assert gpu["kept_count"].tolist() == cpu["kept_count"].tolist()
    parity_util.assert_results_match(gpu, cpu, "f32", "foreseen ends")


@pytest.mark.parametrize("equal", [4097, 8192, 70000])
def test_a_bin_of_more_than_two_to_the_32_steps(equal):
    """A few tokens above thousands of equal ones: the equal ones' steps at the exponent of the sum in front of them add up to
    2^32 and more, which must not be taken for the small number that is left of them modulo 2^32."""
    heights = [np.float32(0.6931472), np.float32(0.0078125), np.float32(2.0), np.float32(8.0), np.float32(16.0)]
    rows, vocab = 2 * len(heights), equal + 3
    print("[case] flat rows of %d with spikes" % equal, flush=True)
    logits = np.zeros((rows, vocab), dtype=np.float32)
    for i, height in enumerate(heights):
        logits[2 * i, vocab // 2] = height
        logits[2 * i + 1, :3] = height
    params = hip_sampler.make_params(rows, 1.0, 0, 1.0, 0.0)
    params["top_p"][1::4] = np.float32(0.7)
    uniforms = np.linspace(0.05, 0.95, rows).astype(np.float32)
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(logits)
        gpu = sampler.sample(params, uniforms)
    assert gpu["kept_count"].tolist() == cpu["kept_count"].tolist()
    parity_util.assert_results_match(gpu, cpu, "f32", "flat rows")


@pytest.mark.parametrize("rows,vocab,finite", [(64, 4096, 4096), (7, 16384, 16384), (5, 100003, 20000)])
def test_runs_of_listed_bins(rows, vocab, finite):
    """Short rows, and rows whose last binades are listed, have long runs of listed bins: the sums end behind them, and at
    stops, windows and cuts inside them."""
    rng = np.random.default_rng(rows + vocab)
    print("[case] runs of listed bins, %d x %d" % (rows, vocab), flush=True)
    logits = np.full((rows, vocab), -np.inf, dtype=np.float32)
    for row in logits:
        row[rng.choice(vocab, finite, replace=False)] = rng.standard_normal(finite) * 2.5
    uniforms = rng.random(rows, dtype=np.float32)
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(logits)
        for top_p, min_p, top_k in ((1.0, 0.0, 0), (0.9999, 0.0, 0), (0.95, 0.0, 0), (1.0, 2e-5, 0), (1.0, 3e-4, 0), (1.0, 0.0, finite // 2), (0.999, 1e-4, finite - 1)):
            params = hip_sampler.make_params(rows, 1.0, top_k, top_p, min_p)
            cpu = parity_util.run_oracle(logits, params, uniforms)
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "top_p %g min_p %g top_k %d" % (top_p, min_p, top_k))


@pytest.mark.parametrize("vocab", [4200, 40003, 151936])
@pytest.mark.parametrize("kind", ["halves", "eighths", "equal", "two values", "equal terms of several logits"])
def test_thousands_of_equal_terms(kind, vocab):
    """Draws, Top-P ends, windows and cuts among thousands of equal terms, at the top of the row and behind it: the token is the
    one of that rank in the row's order, and no row is left to the sort."""
    rng = np.random.default_rng(vocab)
    rows = 10
    print("[case] equal terms, %s x %d" % (kind, vocab), flush=True)
    base = rng.standard_normal((rows, vocab))
    logits = {"halves": np.round(base * 4) / 2, "eighths": np.round(base * 16) / 8, "equal": np.full((rows, vocab), 0.5),
              "two values": (base > 0.5) * 1.5, "equal terms of several logits": rng.integers(0, 6, (rows, vocab)) * 1e-9 + (base > 1.0)}[kind].astype(np.float32)
    uniforms = np.linspace(0.0, 0.97, rows).astype(np.float32)  # (a draw that no partial sum exceeds is the sort's)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.upload_logits(logits)
        for top_p, min_p, top_k in ((0.95, 0.0, 0), (1.0, 0.0, 0), (1.0, 0.01, 0), (0.5, 0.0, vocab // 2), (1e-6, 0.0, 0)):
            params = hip_sampler.make_params(rows, 1.0, top_k, top_p, min_p)
            cpu = parity_util.run_oracle(logits, params, uniforms)
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "%s top_p %g min_p %g top_k %d" % (kind, top_p, min_p, top_k))
            assert sampler.binned_rows(rows).tolist() == [1] * rows, (top_p, min_p, top_k)


@pytest.mark.parametrize("vocab", [4099, 16384])
def test_runs_of_listed_bins_that_end_with_the_sum(vocab):
    """A Min-P cut or a window ends the sum behind a run of listed bins, and the next bins hold nothing: the end is not run past."""
    rng = np.random.default_rng(vocab + 1)
    rows = 64
    print("[case] runs that end with the sum, %d x %d" % (rows, vocab), flush=True)
    logits = _bf16_values((rng.standard_normal((rows, vocab)) * rng.uniform(1.5, 4.0, (rows, 1))).astype(np.float32))
    uniforms = rng.random(rows, dtype=np.float32)
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(logits)
        for top_p, min_p, top_k in ((1.0, 1e-6, 0), (1.0, 3e-6, 0), (1.0, 3e-5, 0), (0.9999, 1e-6, 0), (1.0, 0.0, vocab - 20), (1.0, 1e-6, vocab - 20)):
            params = hip_sampler.make_params(rows, 1.0, top_k, top_p, min_p)
            cpu = parity_util.run_oracle(logits, params, uniforms)
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "top_p %g min_p %g top_k %d" % (top_p, min_p, top_k))


@pytest.mark.parametrize("vocab", [20011, 100003, 151936])
@pytest.mark.parametrize("spread", [0.3, 1.0, 1.33, 1.8, 2.5])
def test_terms_half_way_at_every_distance(spread, vocab):
    """Rows whose sums meet terms that lie half way between two sums 10 to 20 binades below them: those that no mask, a narrow one and a
    wide one tells, in the normaliser, the Top-P sum and the draw.  (Rounded to 1/4096 the rows hold many of them twice.)"""
    rng = np.random.default_rng(int(spread * 100) + vocab)
    rows = 40
    print("[case] terms half way, %d of spread %g" % (vocab, spread), flush=True)
    logits = (rng.standard_normal((rows, vocab)) * spread).astype(np.float32)
    logits[::3] = (np.round(logits[::3] * 4096.0) / 4096.0).astype(np.float32)
    params = hip_sampler.make_params(rows, 1.0, 0, 1.0, 0.0)
    params["temperature"] = rng.choice(np.array([1.0, 0.8, 1.3], dtype=np.float32), rows)
    params["top_p"] = rng.choice(np.array([1.0, 0.9999, 0.99, 0.9, 0.7], dtype=np.float32), rows)
    uniforms = rng.random(rows, dtype=np.float32)
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(logits)
        parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "terms half way, %d of spread %g" % (vocab, spread))


@pytest.mark.parametrize("vocab", [1921, 4096, 8192])
@pytest.mark.parametrize("spread", [1.0, 2.0, 2.5])
def test_heads_that_hold_the_top_p_and_heads_that_end_before_it(spread, vocab):
    """Rows short enough for the longest sorted head to hold the whole Top-P, nearly all of it or less, and draws on both sides of
    the head's end: the head ends early or late by the row's own Top-P, and the token, the filters and the draw stay the same."""
    rng = np.random.default_rng(int(spread * 100) + vocab)
    rows = 48
    print("[case] heads, %d of spread %g" % (vocab, spread), flush=True)
    logits = (rng.standard_normal((rows, vocab)) * spread).astype(np.float32)
    params = hip_sampler.make_params(rows, 1.0, 0, 1.0, 0.0)
    params["top_p"] = np.linspace(0.3, 1.0, rows, dtype=np.float32)
    uniforms = rng.random(rows, dtype=np.float32)
    uniforms[::4] = np.float32(1.0) - np.float32(2.0) ** -24
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(logits)
        parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "heads, %d of spread %g" % (vocab, spread))


@pytest.mark.parametrize("vocab", [1920, 1921, 2047, 2048, 2049, 5000])
def test_rows_and_windows_that_are_all_head(vocab):
    """Rows, finite prefixes and windows of 1,920 to 2,049 elements, which the sorted head holds whole or just does not, with sums
    that run to their ends."""
    rng = np.random.default_rng(vocab + 7)
    rows = 24
    print("[case] all head, %d" % vocab, flush=True)
    logits = (rng.standard_normal((rows, vocab)) * rng.uniform(0.3, 4.0, (rows, 1))).astype(np.float32)
    logits[1::4] = np.round(logits[1::4] * 8) / 8
    logits[2::4] -= np.where(rng.random((rows // 4, vocab)) < 0.1, np.float32(40.0), np.float32(0.0))  # terms that move no sum
    if vocab == 5000:
        logits[3::4, rng.permutation(vocab)[:vocab - 2048]] = -np.inf
    uniforms = rng.random(rows, dtype=np.float32)
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(logits)
        for top_p, min_p, top_k in ((1.0, 0.0, 0), (0.9999, 0.0, 0), (0.9, 0.0, 0), (1.0, 1e-4, 0), (1.0, 0.0, 1921), (1.0, 0.0, 2048), (0.999, 0.0, 2049)):
            params = hip_sampler.make_params(rows, 1.0, top_k, top_p, min_p)
            cpu = parity_util.run_oracle(logits, params, uniforms)
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "all head, %d top_p %g min_p %g top_k %d" % (vocab, top_p, min_p, top_k))


@pytest.mark.parametrize("vocab", [4096, 16384, 32003])
@pytest.mark.parametrize("spread", [1.5, 2.5])
def test_min_p_cuts_around_the_ends_of_heads(spread, vocab):
    """Min-P cuts in front of the head that ends early, between it and the end of the longest one, and behind both."""
    rng = np.random.default_rng(int(spread * 10) + vocab)
    rows = 48
    print("[case] cuts around heads, %d of spread %g" % (vocab, spread), flush=True)
    logits = (rng.standard_normal((rows, vocab)) * spread).astype(np.float32)
    logits[::6] = np.round(logits[::6] * 16) / 16
    params = hip_sampler.make_params(rows, 1.0, 0, 1.0, 0.0)
    params["min_p"] = np.geomspace(3e-4, 0.2, rows).astype(np.float32)
    params["top_p"][1::3] = np.float32(0.9)
    params["top_p"][2::3] = np.float32(0.999)
    uniforms = rng.random(rows, dtype=np.float32)
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        sampler.upload_logits(logits)
        parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "cuts around heads, %d of spread %g" % (vocab, spread))


@pytest.mark.parametrize("first_bin", [3967, 3968, 3969, 4032, 4033, 4095, 4096, 4097])
@pytest.mark.parametrize("behind", [0, 900])
def test_heads_of_one_bin_up_to_the_whole_list(first_bin, behind):
    """A first bin is in the head whatever it holds, up to the list's 4,096 elements: heads that end in the last 64 of them, of
    equal and of unequal terms, with and without elements behind, ended by the row, by Top-P, by Min-P and by the draw."""
    rng = np.random.default_rng(first_bin + behind)
    rows, vocab = 12, first_bin + behind
    print("[case] one bin of %d, %d behind" % (first_bin, behind), flush=True)
    logits = np.full((rows, vocab), 0.5, dtype=np.float32)
    logits[1::2, :first_bin] += rng.random((rows // 2, first_bin), dtype=np.float32) * np.float32(0.003)
    logits[:, first_bin:] -= rng.random((rows, behind), dtype=np.float32) * np.float32(6.0) + np.float32(0.02)
    logits = np.ascontiguousarray(rng.permuted(logits, axis=1))
    uniforms = np.linspace(0.0, 0.97, rows).astype(np.float32)  # (a draw that no partial sum exceeds is the sort's)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.upload_logits(logits)
        for top_p, min_p in ((1.0, 0.0), (0.97, 0.0), (0.5, 0.0), (1.0, 0.99), (1e-6, 0.0)):
            params = hip_sampler.make_params(rows, 1.0, 0, top_p, min_p)
            cpu = parity_util.run_oracle(logits, params, uniforms)
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "one bin of %d, top_p %g min_p %g" % (first_bin, top_p, min_p))
            if first_bin <= 4096:
                assert sampler.binned_rows(rows).tolist() == [1] * rows, (top_p, min_p)


@pytest.mark.parametrize("exponent", [-22, -1, 0, 1, 21])
def test_quotients_of_terms_are_correctly_rounded(exponent):
    """The quotients that the sums add up as whole steps, against numpy's division (correctly rounded): every mantissa of the
    dividend by divisors of the kinds at which a corrected quotient can go wrong (at and next to a power of two, 2/3 and 4/3, sqrt 2,
    the last mantissas) and random ones, then random pairs, over the terms' and divisors' whole range."""
    rng = np.random.default_rng(exponent + 100)
    print("[case] quotients, divisors of 2^%d" % exponent, flush=True)
    mantissas = np.concatenate([np.array([0, 1, 2, 3, 0x7fffff, 0x7ffffe, 0x7ffffd, 0x555555, 0x2aaaab, 0x3504f3, 0x400000], dtype=np.uint32),
                                rng.integers(0, 1 << 23, 5).astype(np.uint32)])
    divisors = ((np.uint32(127 + exponent) << 23) | mantissas).astype(np.uint32).view(np.float32)
    every = np.arange(1 << 23, dtype=np.uint32)
    with hip_sampler.HipSampler(1, 64, testing=True) as sampler:
        for i, divisor in enumerate(divisors):
            term_exponent = -25 + (7 * i) % 25
            dividends = ((np.uint32(127 + term_exponent) << 23) | every).view(np.float32)
            quotients = sampler.quotients(dividends, np.full_like(dividends, divisor))
            wrong = np.nonzero(quotients.view(np.uint32) != (dividends / divisor).view(np.uint32))[0]
            assert wrong.size == 0, "%r / %r" % (dividends[wrong[0]], divisor)
        some = 1 << 23
        dividends = (((127 - rng.integers(0, 26, some)) << 23) | rng.integers(0, 1 << 23, some)).astype(np.uint32).view(np.float32)
        divisors = ((np.uint32(127 + exponent) << 23) | rng.integers(0, 1 << 23, some).astype(np.uint32)).view(np.float32)
        quotients = sampler.quotients(dividends, divisors)
        assert np.array_equal(quotients.view(np.uint32), (dividends / divisors).view(np.uint32))
        # ... and a quotient divided again, as the draw's terms are
        again = (((127 - rng.integers(1, 23, some)) << 23) | rng.integers(0, 1 << 23, some)).astype(np.uint32).view(np.float32)
        if exponent >= 0:
            assert np.array_equal(sampler.quotients(quotients, again).view(np.uint32), (quotients / again).view(np.uint32))


# (a trip of the chain's loads is 8,192 terms, here a sixteenth of the row's; of the four launches' 16,384 in the sum and 8,192 in the walks)
@pytest.mark.parametrize("rows,vocab", [(2, 163839), (2, 163848), (2, 10239), (1, 10249), (260, 4100), (2, 131072), (2, 131080), (260, 8192), (260, 8200),
                                        (260, 16384), (260, 16392)])
def test_steps_at_the_ends_of_their_trips(rows, vocab):
    """Parts that take one trip of their terms' loads and one group of eight more, in one launch and in four: logits of eighths, whose equal terms and terms
    half way between two sums reach every kind of bin, beside plain ones."""
    rng = np.random.default_rng(rows * 7 + vocab)
    print("[case] trips of steps, %d x %d" % (rows, vocab), flush=True)
    logits = (rng.standard_normal((rows, vocab)) * 2.5).astype(np.float32)
    logits[::2] = np.round(logits[::2] * 8) / 8
    params = hip_sampler.make_params(rows, 1.0, 0, 0.999, 0.0)
    params["top_p"][1::2] = 1.0
    uniforms = rng.random(rows, dtype=np.float32)
    uniforms[-1] = np.float32(0.9999)
    cpu = parity_util.run_oracle(logits, params, uniforms)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        sampler.binned_sums(True)
        sampler.upload_logits(logits)
        gpu = sampler.sample(params, uniforms)
    parity_util.assert_results_match(gpu, cpu, "f32", "trips of steps")
