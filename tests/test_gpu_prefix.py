"""The prefix-sort path at the sizes and structures where its steps change: one and two bucket
levels, samples sorted in one workgroup and by radix, skewed keys, leaves beyond the LDS, small and
large tie groups, alphabets of 1 to 9 bits, batches whose texts have their own codes. Every row of
the suffix array and every BWT byte is checked on the device; small texts against the oracle too."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def text_of(kind, n):
    from sadcs_amd import workloads
    rng = np.random.default_rng(n + len(kind))
    if kind in ("dna_uniform", "dna_like", "markov", "protein", "periodic"):
        return getattr(workloads, kind)(n, seed=n & 1023)
    if kind == "bytes":
        return rng.integers(0, 256, n, dtype=np.uint8)
    if kind == "zeros":  # long runs of one byte between rare others: skewed keys, large groups
        return (rng.random(n) < 0.02).astype(np.uint8) * rng.integers(1, 4, n, dtype=np.uint8)
    if kind == "runs":  # DNA with runs: leaves of equal keys, beyond the LDS from 100,000 bytes on
        t = workloads.dna_uniform(n, seed=3)
        for _ in range(6):
            at = int(rng.integers(0, n - n // 100))
            t[at:at + n // 100] = ord("N")
        return t
    if kind == "copies":  # one piece 40 times among random text: groups larger than the LDS compares
        t = rng.integers(0, 200, n, dtype=np.uint8)
        piece = rng.integers(0, 200, max(8, n // 2000), dtype=np.uint8)
        for at in rng.integers(0, n - piece.size, 40):
            t[at:at + piece.size] = piece
        return t
    assert kind == "pairs"  # half of the text is a copy of the other half
    half = workloads.protein((n + 1) // 2, seed=9)
    return np.concatenate([half, half])[:n]


def check_device(gpu, text, cover=32, want_sa=True, want_bwt=True):
    n = text.size
    d_text = gpu.DeviceBuffer.from_host(np.ascontiguousarray(text), extra=64)
    d_sa, d_bwt = gpu.DeviceBuffer(4 * n), gpu.DeviceBuffer(n)
    with gpu.GpuContext(n, cover=cover) as ctx:
        primary = gpu.gpu_build_device(ctx, d_text.ptr, n, d_sa.ptr, d_bwt.ptr)
        assert gpu.gpu_check_device(d_text.ptr, n, d_sa.ptr, d_bwt.ptr, primary) == (0, -1)
        sa, bwt = d_sa.to_host(np.int32), d_bwt.to_host(np.uint8).tobytes()
        d_one = gpu.DeviceBuffer(4 * n)
        gpu.gpu_build_device(ctx, d_text.ptr, n, d_one.ptr, None)
        assert np.array_equal(d_one.to_host(np.int32), sa)
        d_one = gpu.DeviceBuffer(n)
        assert gpu.gpu_build_device(ctx, d_text.ptr, n, None, d_one.ptr) == primary
        assert d_one.to_host(np.uint8).tobytes() == bwt
    return sa, bwt, primary


KINDS = ["dna_uniform", "dna_like", "markov", "protein", "periodic", "bytes", "zeros", "runs", "copies", "pairs"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [16385, 65536, 200_001])
def test_prefix_small(gpu, kind, n):
    text = text_of(kind, n)
    sa, bwt, primary = check_device(gpu, text)
    want = oracle.suffix_array(text.tobytes())
    assert np.array_equal(sa, want)
    assert (bwt, primary) == oracle.bwt_from_sa(text.tobytes(), want)
    got = gpu.gpu_build(text, True, True)
    assert np.array_equal(got[0], want) and got[1:] == (bwt, primary)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,cover", [(524_288, 32), (1_050_000, 128), (5_000_003, 32), (20_000_017, 128)])
def test_prefix_large(gpu, kind, n, cover):
    check_device(gpu, text_of(kind, n), cover)


@pytest.mark.parametrize("run", [700, 2047, 3900])
def test_prefix_leaf_spanning_first_bits(gpu, run):
    # Letters 3 and 4 of 8: keys 011... and 100... share a leaf, so its values hold no last four bits,
    # and a run's keys differ in those alone.
    rng = np.random.default_rng(run)
    text = rng.integers(0, 8, 20_000 + run, dtype=np.uint8)
    text[5000:5000 + run] = 3
    text[15000:15000 + run // 2] = 4
    for at in range(5000 + 16, 5000 + run, 400):  # breaks: a key's 18 letters end before, at and behind
        text[at] = rng.integers(0, 8)
    sa, bwt, primary = check_device(gpu, text)
    want = oracle.suffix_array(text.tobytes())
    assert np.array_equal(sa, want)
    assert (bwt, primary) == oracle.bwt_from_sa(text.tobytes(), want)


def test_prefix_batches(gpu):
    from sadcs_amd import workloads
    rng = np.random.default_rng(5)
    # Texts that end just before a 256-boundary, where the next text (of other codes) starts.
    close = [256 * k - d for k, d in zip(range(70, 130), [0, 1, 2, 3, 7, 8, 9, 15, 16, 17, 23, 24] * 5)]
    for sizes in ([20_000, 1, 256, 257, 70_000, 255], [300_000] * 3 + [5, 4096], close, rng.integers(1, 60_000, 200).tolist() + [3_000_000]):
        texts = [text_of(KINDS[i % len(KINDS)], max(n, 300))[:n] for i, n in enumerate(sizes)]
        lengths = np.array([t.size for t in texts], dtype=np.int64)
        offsets, span = gpu.gpu_batch_layout(lengths)
        host = np.zeros(span + 64, dtype=np.uint8)
        for t, o in zip(texts, offsets.tolist()):
            host[o:o + t.size] = t
        d_texts = gpu.DeviceBuffer.from_host(host)
        total = int(lengths.sum())
        d_sa, d_bwt = gpu.DeviceBuffer(4 * total), gpu.DeviceBuffer(total)
        with gpu.GpuContext(0, batch_lengths=lengths) as ctx:
            primaries = gpu.gpu_batch_build_device(ctx, d_texts.ptr, lengths, d_sa.ptr, d_bwt.ptr)
            d_one = gpu.DeviceBuffer(total)
            assert np.array_equal(gpu.gpu_batch_build_device(ctx, d_texts.ptr, lengths, None, d_one.ptr), primaries)
        assert np.array_equal(d_one.to_host(np.uint8), d_bwt.to_host(np.uint8))
        at = 0
        for i, t in enumerate(texts):
            result = gpu.gpu_check_device(d_texts.ptr + int(offsets[i]), t.size, d_sa.ptr + 4 * at, d_bwt.ptr + at, int(primaries[i]))
            assert result == (0, -1), f"text {i} of {t.size} bytes"
            at += t.size


def test_host_batch_gathered_in_pieces(gpu):
    # Texts that end before, at and past the 2 MiB pieces of the upload, and one over three of them.
    from sadcs_amd import workloads
    mib = 1 << 20
    lengths = [2 * mib - 100, 2 * mib, 300, 2 * mib - 512 + 1, 70_000, 1, 4 * mib + 255, 20_000]
    texts = [workloads.protein(n, seed=n & 1023) for n in lengths]
    for text, (sa, bwt, primary) in zip(texts, gpu.gpu_batch_build(texts, True, True)):
        want = gpu.gpu_build(text, True, True)
        assert np.array_equal(sa, want[0]) and (bwt, primary) == want[1:]


@pytest.mark.parametrize("n", [4096 - 7, 4096, 4096 + 9, 8192 + 1, 12_288 - 5, 33_000, 65_536 + 40, 300_007, 2_097_152 + 16, 2_200_000])
def test_sample_sorted_by_merges(gpu, n):
    # The ranking sorts about n / 4 sample keys: under, at and over the chunks that a workgroup sorts,
    # odd numbers of runs, and over the length from which digit passes take them. The suffix array that
    # the ranks imply comes from another path.
    from sadcs_amd import workloads
    for text in (workloads.dna_like(n, seed=5), workloads.periodic(n, seed=6)):
        sa, _, _ = check_device(gpu, text)
        assert np.array_equal(gpu.gpu_rank_sample(text), oracle.sample_ranks_from_sa(sa, 32))


@pytest.mark.parametrize("n", [16_385, 118_796, 1_048_577, 5_000_011])
def test_cover_128_by_cover_32(gpu, n):
    # Texts that the prefix sort leaves to the tile merge: a context of cover 128 with room for it takes
    # cover 32, one with merge parameters its own.
    for kind in ("periodic", "zeros"):
        text = text_of(kind, n)
        d_text = gpu.DeviceBuffer.from_host(text, extra=64)
        d_sa, d_bwt = gpu.DeviceBuffer(4 * n), gpu.DeviceBuffer(n)
        with gpu.GpuContext(n, cover=128, tile_splitters=8) as ctx:
            primary = gpu.gpu_build_device(ctx, d_text.ptr, n, d_sa.ptr, d_bwt.ptr)
        assert gpu.gpu_check_device(d_text.ptr, n, d_sa.ptr, d_bwt.ptr, primary) == (0, -1)
        sa, bwt, got = check_device(gpu, text, cover=128)
        assert np.array_equal(sa, d_sa.to_host(np.int32)) and bwt == d_bwt.to_host(np.uint8).tobytes() and got == primary


@pytest.mark.parametrize("n", [700_001, (1 << 20) - 1])
def test_short_text_in_what_a_longer_one_needs(gpu, n):
    # A context with merge parameters holds its plan and no more; a server's budget of twelve bytes a byte
    # leaves nothing beyond the plan. Both take the text, as does a context of its own.
    text = text_of("protein", n)
    want, bwt, primary = check_device(gpu, text)
    with gpu.GpuContext(1 << 20, tile_splitters=8) as ctx:
        sa, b, p = gpu.gpu_build(text, True, True, context=ctx)
    assert np.array_equal(sa, want) and (b, p) == (bwt, primary)
    with gpu.Server(memory_budget=12 << 20, workers=1) as server:
        sa, b, p, *_ = server.wait(server.submit(text))
    assert np.array_equal(sa, want) and (b, p) == (bwt, primary)
    sa, b, p = gpu.gpu_build(text, True, True)
    assert np.array_equal(sa, want) and (b, p) == (bwt, primary)
