"""The tile merge as its own path, at both covers: contexts with merge parameters (the covers' defaults,
given) take it for every text, also for those that the other paths build by default."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

PARAMS = {32: {"splitter_spacing": 16}, 128: {"cover": 128, "splitter_spacing": 8}}


def small_texts():
    rng = oracle.Rng(31)
    yield from (b"a", b"ab", b"banana", b"mississippi", b"\xff" * 1000, b"\0" * 999 + b"\1", bytes(range(256)) * 3)
    for n in (31, 32, 33, 64, 127, 129, 4097, 16_384):
        yield from (rng.random_text(n, 4), rng.random_text(n, 256), rng.periodic_text(n, 33))
    yield oracle.fibonacci_text(10_000)
    yield oracle.thue_morse_text(8192)


@pytest.mark.parametrize("cover", [32, 128])
def test_small_texts(gpu, cover):
    texts = list(small_texts())
    with gpu.GpuContext(1 << 15, **PARAMS[cover]) as ctx:
        for text in texts:
            want = oracle.naive_sa(text)
            bwt = oracle.bwt_from_sa(text, want)
            sa, b, primary = gpu.gpu_build(text, True, True, context=ctx)  # the fused merge
            assert np.array_equal(sa, want) and (b, primary) == bwt, len(text)
            assert np.array_equal(gpu.gpu_suffix_array(text, context=ctx), want) and gpu.gpu_bwt(text, context=ctx) == bwt, len(text)
    with gpu.GpuContext(0, batch_lengths=[len(t) for t in texts], **PARAMS[cover]) as ctx:
        for text, (sa, b, primary) in zip(texts, gpu.gpu_batch_build(texts, context=ctx)):
            want = oracle.naive_sa(text)
            assert np.array_equal(sa, want) and (b, primary) == oracle.bwt_from_sa(text, want), len(text)


@pytest.mark.parametrize("cover", [32, 128])
@pytest.mark.parametrize("kind", ["dna_like", "markov"])
def test_repeated_fused_builds(gpu, kind, cover):
    """Texts with long repeats: many comparisons past the records' 32 characters and down to the ranks."""
    from sadcs_amd import workloads
    text = getattr(workloads, kind)(3 << 20, seed=43).tobytes()
    want = oracle.suffix_array(text)
    want_bwt = oracle.bwt_from_sa(text, want)
    with gpu.GpuContext(len(text), **PARAMS[cover]) as ctx:
        for r in range(4):
            print(f"cover {cover} fused {kind} build {r}", flush=True)
            sa, b, primary = gpu.gpu_build(text, True, True, context=ctx)
            assert np.array_equal(sa, want) and (b, primary) == want_bwt, r
