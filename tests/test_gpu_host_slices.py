"""Host calls of more than 2^24 rows whose outputs are downloaded in row slices while the tile merge runs:
contexts with merge parameters, texts that the prefix sort leaves to the merge, and long texts whose suffix
array is asked for. Whatever the slicing, they return what a device-resident build, checked row by
row, leaves in HBM."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MiB = 1 << 20
OUTPUTS = [(True, True), (True, False), (False, True)]


def text_of(kind, n):
    from sadcs_amd import workloads
    return getattr(workloads, kind)(n, seed=n & 255)


def device_build(gpu, text):
    n = text.size
    d_text, d_sa, d_bwt = gpu.DeviceBuffer.from_host(text, extra=64), gpu.DeviceBuffer(4 * n), gpu.DeviceBuffer(n)
    with gpu.GpuContext(n) as ctx:
        primary = gpu.gpu_build_device(ctx, d_text.ptr, n, d_sa.ptr, d_bwt.ptr)
    assert gpu.gpu_check_device(d_text.ptr, n, d_sa.ptr, d_bwt.ptr, primary) == (0, -1)
    outputs = d_sa.to_host(np.int32), d_bwt.to_host(np.uint8), primary
    for buffer in (d_text, d_sa, d_bwt):
        buffer.free()
    return outputs


def host_build(gpu, ctx, text, sa, bwt, sa_ptr, bwt_ptr):
    primary = ctypes.c_int32(-1)
    status = gpu.lib.sadcs_hip_build(ctx.handle, text, sa.size if sa is not None else bwt.size, sa_ptr if sa is not None else None,
                                     bwt_ptr if bwt is not None else None, ctypes.byref(primary), None)
    assert status == 0, gpu.gpu_last_error()
    return primary.value


CASES = [("markov", 40 * MiB, {"splitter_spacing": 16}), ("dna_like", (1 << 24) + 12_345, {"tile_splitters": 40}),
         ("markov", 40 * MiB, {"cover": 128, "splitter_spacing": 8}), ("periodic", (1 << 24) + 12_345, {}),
         ("dna_like", 48 * MiB + 1, {}), ("markov", 75 * MiB + 77, {}), ("protein", 50 * MiB, {"cover": 128})]


@pytest.mark.parametrize("kind,n,params", CASES, ids=[f"{k}-{n}-{'-'.join(f'{a}{b}' for a, b in p.items()) or 'default'}" for k, n, p in CASES])
@pytest.mark.parametrize("pinned", [False, True], ids=["pageable", "pinned"])
def test_host_call_in_slices(gpu, kind, n, params, pinned):
    text = text_of(kind, n)
    want_sa, want_bwt, want_primary = device_build(gpu, text)
    pointers = []
    if pinned:
        (sa_ptr, sa_view), (bwt_ptr, bwt_view) = gpu.gpu_allocate_pinned(4 * n), gpu.gpu_allocate_pinned(n)
        pointers = [sa_ptr, bwt_ptr]
        sa, bwt = sa_view.view(np.int32), bwt_view
    else:
        sa, bwt = np.empty(n, dtype=np.int32), np.empty(n, dtype=np.uint8)
        sa_ptr, bwt_ptr = sa.ctypes.data, bwt.ctypes.data
    try:
        with gpu.GpuContext(n, **params) as ctx:
            for with_sa, with_bwt in OUTPUTS:
                print(f"{kind} {n} {params} sa={with_sa} bwt={with_bwt}", flush=True)
                sa[:] = -1
                bwt[:] = 0xEE
                primary = host_build(gpu, ctx, text.ctypes.data, sa if with_sa else None, bwt if with_bwt else None, sa_ptr, bwt_ptr)
                assert not with_sa or np.array_equal(sa, want_sa)
                assert not with_bwt or (np.array_equal(bwt, want_bwt) and primary == want_primary)
    finally:
        for pointer in pointers:
            gpu.gpu_free_pinned(pointer)


@pytest.mark.parametrize("params", [{"splitter_spacing": 16}, {}], ids=["merge parameters", "default"])
def test_host_batch_in_slices(gpu, params):
    """Slices that cut across texts: every text's rows and bytes equal its own device-resident build's."""
    rng = np.random.default_rng(12)
    lengths = [int(x) for x in rng.integers(1 * MiB, 4 * MiB, 22)]
    texts = [text_of(("markov", "dna_like", "protein")[i % 3], n) for i, n in enumerate(lengths)]
    assert sum(lengths) > 48 * MiB
    with gpu.GpuContext(0, batch_lengths=lengths, **params) as ctx:
        both = gpu.gpu_batch_build(texts, context=ctx)
        alone = gpu.gpu_batch_build(texts, True, False, context=ctx)
    for text, (sa, bwt, primary), (sa_alone, _, _) in zip(texts, both, alone):
        want = device_build(gpu, text)
        assert np.array_equal(sa, want[0]) and np.array_equal(sa_alone, want[0])
        assert bwt == want[1].tobytes() and primary == want[2]


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
