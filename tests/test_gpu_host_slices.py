"""Which path a host call takes, and with it whether its outputs are downloaded while it runs."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MiB = 1 << 20


def text_of(kind, n):
    from sadcs_amd import workloads
    return getattr(workloads, kind)(n, seed=n & 255)


@pytest.mark.parametrize("n,sa,merge", [(48 * MiB, True, False), (48 * MiB + 1, True, True), (64 * MiB, True, True), (64 * MiB, False, False)])
def test_path_of_a_long_host_call(gpu, n, sa, merge):
    """More than 48 MiB of text whose suffix array goes to the host take the tile merge, which downloads while
    it merges: the call's memory, phase by phase, is that of a context with the merge's default parameters."""
    text = text_of("dna_like", n)
    outputs = [np.empty(n, dtype=np.int32) if sa else None, np.empty(n, dtype=np.uint8)]
    used = []
    for params in ({}, {"splitter_spacing": 16}):
        stats, primary = gpu.GpuStats(), ctypes.c_int32(-1)
        with gpu.GpuContext(n, **params) as ctx:
            assert gpu.lib.sadcs_hip_build(ctx.handle, text.ctypes.data, n, outputs[0].ctypes.data if sa else None, outputs[1].ctypes.data,
                                           ctypes.byref(primary), ctypes.byref(stats)) == 0
        used.append((stats.ranking_bytes, stats.class_sort_bytes, stats.merge_bytes))
        print(f"{n} sa={sa} {params}: {used[-1]}, upload {stats.upload_seconds * 1e3:.1f}, device {stats.device_seconds * 1e3:.1f}, "
              f"download {stats.download_seconds * 1e3:.1f} ms", flush=True)
    assert (used[0] == used[1]) == merge
