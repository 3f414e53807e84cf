"""ncnn_moe_hip_sampler_upload_logits: what arrives in the handle's buffer is what the host held, word for word, for uploads that are
one piece and several, end on both sides of a piece and of what the pinned staging holds, and come from rows that are further apart; also
behind an error that an earlier call left, behind long work, and on a handle whose calls are replayed from a graph."""
import time

import numpy as np
import pytest

import parity_util
from ncnn_moe_runtime_amd import hip_sampler

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

PIECE = 320 << 10
STAGING = 4 << 20


class _DeviceWords:
    def __init__(self, pointer, count):
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<i2", "data": (pointer, False), "version": 2}


def _in_device(sampler, dtype, rows, vocab, halves):
    """[rows, vocab] as 16-bit words of the handle's buffer."""
    pointer, stride = sampler.logits_buffer(dtype, rows, vocab)
    words = torch.as_tensor(_DeviceWords(pointer, rows * stride * halves), device="cuda:0").cpu().numpy()
    return words.reshape(rows, stride * halves)[:, :vocab * halves]


SHAPES = [(1, 1), (1, 7), (3, 5), (1, PIECE // 4), (1, PIECE // 4 + 1), (2, PIECE // 2 + 3), (5, PIECE // 4 - 1), (16, STAGING // 64), (16, STAGING // 64 + 1), (7, 100003)]


@pytest.mark.parametrize("rows,vocab", SHAPES)
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("pinned", [False, True])
def test_uploads_arrive_whole(rows, vocab, bf16, pinned):
    print("[case] upload %d x %d, bf16 %s, pinned %s" % (rows, vocab, bf16, pinned), flush=True)
    rng = np.random.default_rng(rows * 131 + vocab)
    dtype = hip_sampler.LOGITS_BF16 if bf16 else hip_sampler.LOGITS_F32
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        for apart in (0, 3):
            for _ in range(2):
                held = torch.from_numpy(rng.integers(0, 1 << 15, (rows, (vocab + apart) * (1 if bf16 else 2)), dtype=np.int16))
                held = held.pin_memory() if pinned else held
                logits = held.numpy().view(np.uint16 if bf16 else np.float32)
                sampler.upload_logits(logits, vocab)
                halves = 1 if bf16 else 2
                assert np.array_equal(_in_device(sampler, dtype, rows, vocab, halves), held.numpy()[:, :vocab * halves])


def test_uploads_and_calls_on_other_streams_in_turn():
    """Upload, sample on the handle's stream, upload again and sample_device on another one from the handle's buffer."""
    rows, vocab = 3, 50257
    rng = np.random.default_rng(5)
    params = hip_sampler.make_params(rows, 0.8, 20, 0.9, 0.0)
    uniforms = rng.random(rows, dtype=np.float32)
    on_device = [torch.from_numpy(x.view(np.uint8).copy()).cuda() for x in (params, uniforms)]
    results = torch.zeros(rows * 16, dtype=torch.uint8, device="cuda:0")
    stream = torch.cuda.Stream()
    with hip_sampler.HipSampler(rows, vocab) as sampler:
        for turn in range(6):
            print("[case] uploads in turn, %d" % turn, flush=True)
            logits = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
            cpu = parity_util.run_oracle(logits, params, uniforms)
            sampler.upload_logits(logits)
            if turn % 2 == 0:
                gpu = sampler.sample(params, uniforms)
            else:
                pointer, stride = sampler.logits_buffer(hip_sampler.LOGITS_F32, rows, vocab)
                sampler.sample_device(pointer, hip_sampler.LOGITS_F32, rows, vocab, stride, on_device[0].data_ptr(), on_device[1].data_ptr(), None,
                                      results.data_ptr(), 0, stream.cuda_stream)
                stream.synchronize()
                gpu = results.cpu().numpy().view(hip_sampler.RESULT_DTYPE).reshape(rows)
            parity_util.assert_results_match(gpu, cpu, "f32", "turn %d" % turn)


@pytest.mark.parametrize("rows,vocab", [(1, 7), (4, PIECE // 4)])
def test_an_error_that_an_earlier_call_left_is_not_the_uploads(rows, vocab):
    """A device that there is not leaves an error on the thread; the uploads behind it succeed, and the calls behind them read all rows."""
    print("[case] upload %d x %d behind an error" % (rows, vocab), flush=True)
    rng = np.random.default_rng(rows + vocab)
    params = hip_sampler.make_params(rows, 0.8, min(20, vocab), 0.9, 0.0)
    uniforms = rng.random(rows, dtype=np.float32)
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        for _ in range(3):
            logits = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
            assert sampler._lib.hipSetDevice(1 << 20) != 0
            sampler.upload_logits(logits)
            assert not sampler.stream_may_run()
            cpu = parity_util.run_oracle(logits, params, uniforms)
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "behind an error")


@pytest.mark.parametrize("rows,vocab", [(1, 2003), (4, PIECE // 4)])
def test_uploads_behind_work_that_takes_longer_than_the_host_watches(rows, vocab):
    """The handle's stream waits for the default one: an upload behind some milliseconds of work there is waited for by the stream."""
    print("[case] upload %d x %d behind long work" % (rows, vocab), flush=True)
    rng = np.random.default_rng(rows + vocab)
    halves = 2
    factor = torch.randn(8192, 8192, device="cuda:0")
    product = factor @ factor
    torch.cuda.synchronize()
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        for _ in range(2):
            logits = rng.integers(0, 1 << 15, (rows, vocab * halves), dtype=np.int16)
            for _ in range(4):  # (4.4 TFLOP: 25 ms and more at this card's rate in fp32)
                torch.mm(factor, factor, out=product)
            start = time.perf_counter()
            sampler.upload_logits(logits.view(np.float32), vocab)
            assert time.perf_counter() - start > 0.002
            assert not sampler.stream_may_run()
            assert np.array_equal(_in_device(sampler, hip_sampler.LOGITS_F32, rows, vocab, halves), logits)


def test_uploads_between_replays_of_a_captured_call():
    """sample_device from the handle's buffer, captured, and replayed behind uploads of other logits."""
    rows, vocab = 3, 50257
    rng = np.random.default_rng(9)
    params = hip_sampler.make_params(rows, 0.8, 20, 0.9, 0.0)
    uniforms = rng.random(rows, dtype=np.float32)
    on_device = [torch.from_numpy(x.view(np.uint8).copy()).cuda() for x in (params, uniforms)]
    results = torch.zeros(rows * 16, dtype=torch.uint8, device="cuda:0")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with hip_sampler.HipSampler(rows, vocab, testing=True) as sampler:
        pointer, stride = sampler.logits_buffer(hip_sampler.LOGITS_F32, rows, vocab)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            sampler.sample_device(pointer, hip_sampler.LOGITS_F32, rows, vocab, stride, on_device[0].data_ptr(), on_device[1].data_ptr(), None,
                                  results.data_ptr(), 0, stream.cuda_stream)
        for replay in range(4):
            print("[case] upload and replay, %d" % replay, flush=True)
            logits = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
            cpu = parity_util.run_oracle(logits, params, uniforms)
            sampler.upload_logits(logits)
            assert not sampler.stream_may_run()
            with torch.cuda.stream(stream):
                graph.replay()
            stream.synchronize()
            gpu = results.cpu().numpy().view(hip_sampler.RESULT_DTYPE).reshape(rows)
            parity_util.assert_results_match(gpu, cpu, "f32", "replay %d" % replay)
            parity_util.assert_results_match(sampler.sample(params, uniforms), cpu, "f32", "beside replay %d" % replay)
            results.zero_()
            torch.cuda.synchronize()
