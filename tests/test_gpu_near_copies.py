"""Collections of near-copies (versions of one document, genomes of one species), whole or as part of a text:
groups of tied suffixes of every size. Every row is checked on the device, and the call does not lose to
the tile merge of the same text by more than its look at a sample."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def near_copies(copies, size, seed):
    from sadcs_amd import workloads
    rng = np.random.default_rng(seed)
    text = np.tile(workloads.protein(size, seed=seed), copies)
    at = rng.integers(0, text.size, text.size // 1000)
    text[at] = text[rng.integers(0, size, at.size)]
    return text


def text_of(copies, n, share):
    from sadcs_amd import workloads
    text = workloads.protein(n, seed=5)
    part = near_copies(copies, int(n * share) // copies, copies)
    text[:part.size] = part
    return text


def build(gpu, text, repeats=4, **params):
    """Best milliseconds of a device-resident build, its outputs and its statistics."""
    n = text.size
    d_text, d_sa, d_bwt = gpu.DeviceBuffer.from_host(text, extra=64), gpu.DeviceBuffer(4 * n), gpu.DeviceBuffer(n)
    best, stats = 1e9, gpu.GpuStats()
    with gpu.GpuContext(n, **params) as ctx:
        for _ in range(repeats):
            start = time.perf_counter()
            primary = gpu.gpu_build_device(ctx, d_text.ptr, n, d_sa.ptr, d_bwt.ptr, stats)
            best = min(best, time.perf_counter() - start)
    assert gpu.gpu_check_device(d_text.ptr, n, d_sa.ptr, d_bwt.ptr, primary) == (0, -1)
    outputs = d_sa.to_host(np.int32), d_bwt.to_host(np.uint8), primary
    for buffer in (d_text, d_sa, d_bwt):
        buffer.free()
    return best * 1e3, outputs, stats


@pytest.mark.parametrize("copies", [2, 8, 23, 24, 25, 32, 64, 300])
@pytest.mark.parametrize("n,share", [(60_000, 1.0), (700_000, 0.3), (5_000_000, 1.0), (20_000_000, 0.1)])
def test_near_copies(gpu, copies, n, share):
    text = text_of(copies, n, share)
    _, got, _ = build(gpu, text, repeats=1)
    _, want, _ = build(gpu, text, repeats=1, tile_splitters=8)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]) and got[2] == want[2]


@pytest.mark.parametrize("copies,n,share", [(2, 400 << 20, 1.0), (8, 256 << 20, 1.0), (64, 64 << 20, 1.0), (300, 64 << 20, 1.0),
                                            (64, 256 << 20, 0.1), (64, 256 << 20, 0.35), (64, 48 << 20, 0.5), (64, 4 << 20, 1.0)])
def test_near_copies_against_the_tile_merge(gpu, copies, n, share):
    # The sample costs up to 2% of the merge and 0.1 ms of launches; timing as much again.
    text = text_of(copies, n, share)
    print(f"{copies} copies, {share} of {n} bytes", flush=True)
    ms, got, _ = build(gpu, text)
    tiles, want, _ = build(gpu, text, splitter_spacing=16)  # its default parameters
    print(f"default {ms:.2f} ms, tile merge {tiles:.2f} ms", flush=True)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]) and got[2] == want[2]
    assert ms < 1.05 * tiles + 0.2
