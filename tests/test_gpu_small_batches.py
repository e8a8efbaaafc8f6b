"""Batches of many short texts, one workgroup a text: their statistics, and that they do not lose to the
tile merge of the same batch."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_doubling_rounds_of_a_batch(gpu):
    # 3000 equal bytes: 48 bits of one a character sort by 48 characters, and six doublings pass 3000;
    # 300 take 40 characters and three. The other texts need none.
    rng = np.random.default_rng(1)
    texts = [rng.integers(0, 256, 700, dtype=np.uint8), np.full(300, 7, dtype=np.uint8), rng.integers(0, 256, 90, dtype=np.uint8)]
    for more, rounds in (([], 3), ([np.full(3000, 200, dtype=np.uint8)], 6)):
        stats = gpu.GpuStats()
        gpu.gpu_batch_build(texts + more, stats=stats)
        assert stats.doubling_rounds == rounds


def best_ms(gpu, lengths, **params):
    from sadcs_amd import workloads
    lengths = np.array(lengths, dtype=np.int64)
    offsets, span = gpu.gpu_batch_layout(lengths)
    host = np.zeros(span + 64, dtype=np.uint8)
    source = workloads.markov(int(lengths.sum()), seed=4)
    at = 0
    for n, o in zip(lengths.tolist(), offsets.tolist()):
        host[o:o + n] = source[at:at + n]
        at += n
    d_texts, d_sa, d_bwt = gpu.DeviceBuffer.from_host(host), gpu.DeviceBuffer(4 * at), gpu.DeviceBuffer(at)
    best = 1e9
    with gpu.GpuContext(0, batch_lengths=lengths, **params) as ctx:
        for _ in range(6):
            start = time.perf_counter()
            gpu.gpu_batch_build_device(ctx, d_texts.ptr, lengths, d_sa.ptr, d_bwt.ptr)
            best = min(best, time.perf_counter() - start)
    outputs = d_sa.to_host(np.int32), d_bwt.to_host(np.uint8)
    for buffer in (d_texts, d_sa, d_bwt):
        buffer.free()
    return best * 1e3, outputs


@pytest.mark.parametrize("lengths", [[1024] * 16_000, [100] * 100_000 + [16_384], [16_384, 2049] + [2048, 1] * 1024, [300] * 2047 + [5000]],
                         ids=["16000 of 1 KiB", "100000 of 100 B and one of 16 KiB", "2048 short, two long", "2047 short, one long"])
def test_many_short_texts_against_the_tile_merge(gpu, lengths):
    small, outputs = best_ms(gpu, lengths)
    tiles, want = best_ms(gpu, lengths, splitter_spacing=16)  # its default parameters
    assert np.array_equal(outputs[0], want[0]) and np.array_equal(outputs[1], want[1])
    print(f"one workgroup a text {small:.2f} ms, tile merge {tiles:.2f} ms", flush=True)
    assert small < tiles
