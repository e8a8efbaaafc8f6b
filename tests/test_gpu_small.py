"""Texts one workgroup builds in LDS (up to 16384 bytes), at the edges of its tiles and digits:
every output equals the naive suffix array's, alone and in a batch, on the host and the device."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 63, 64, 65, 255, 256, 257, 1023, 2047, 2048, 2049, 4099, 8192, 16383, 16384, 16385]


def texts_of(n):
    rng = oracle.Rng(100 + n)
    yield "run", b"\xff" * n
    yield "zeros and a one", b"\0" * (n - 1) + b"\1"
    yield "all bytes", rng.random_text(n, 256)
    yield "dna", rng.random_text(n, 4)
    yield "binary", rng.random_text(n, 2)
    yield "period 7", (b"\0ab\0\0b\xff" * (n // 7 + 1))[:n]
    yield "half twice", (rng.random_text((n + 1) // 2, 4) * 2)[:n]


@pytest.mark.parametrize("n", SIZES)
def test_small_alone(gpu, n):
    for name, text in texts_of(n):
        want = oracle.naive_sa(text)
        bwt, primary = oracle.bwt_from_sa(text, want)
        sa, b, p = gpu.gpu_build(text, True, True)
        assert np.array_equal(sa, want) and (b, p) == (bwt, primary), f"{name} n={n}"
        assert np.array_equal(gpu.gpu_suffix_array(text), want), f"{name} n={n}: SA only"
        assert gpu.gpu_bwt(text) == (bwt, primary), f"{name} n={n}: BWT only"


def test_small_batches(gpu):
    """Batches whose outputs pass through pinned memory (short) and through device memory, and one
    on the device at odd output offsets."""
    for sizes in ([1, 5, 64, 256, 257], [2048, 1, 300], SIZES[:-1]):
        texts = [t for n in sizes for _, t in texts_of(n)]
        want = [oracle.naive_sa(t) for t in texts]
        for (sa, b, p), t, w in zip(gpu.gpu_batch_build(texts), texts, want):
            assert np.array_equal(sa, w) and (b, p) == oracle.bwt_from_sa(t, w), f"n={len(t)}"
        lengths = np.array([len(t) for t in texts], dtype=np.int64)
        offsets, span = gpu.gpu_batch_layout(lengths)
        host = np.full(span + 64, 7, dtype=np.uint8)
        for t, o in zip(texts, offsets.tolist()):
            host[o:o + len(t)] = np.frombuffer(t, dtype=np.uint8)
        d_text = gpu.DeviceBuffer.from_host(host)
        total = int(lengths.sum())
        d_sa, d_bwt = gpu.DeviceBuffer(4 * total + 4), gpu.DeviceBuffer(total + 3)
        primaries = gpu.gpu_batch_build_device(None, d_text.ptr, lengths, d_sa.ptr + 4, d_bwt.ptr + 3)
        got_sa, got_bwt, at = d_sa.to_host(np.int32)[1:], d_bwt.to_host(np.uint8)[3:], 0
        for i, (t, w) in enumerate(zip(texts, want)):
            assert np.array_equal(got_sa[at:at + len(t)], w), f"device batch n={len(t)}"
            assert (got_bwt[at:at + len(t)].tobytes(), primaries[i]) == oracle.bwt_from_sa(t, w), f"device batch n={len(t)}"
            at += len(t)
