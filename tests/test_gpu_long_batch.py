"""A long text in a batch: where the characters left in it times the bits of one pass 2^32, near its
start. Every row of the suffix arrays and every BWT byte is checked on the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n", [("markov", 620_000_001), ("bytes", 480_000_003)])  # 7 and 9 bits a character
def test_batch_with_a_long_text(gpu, kind, n):
    from sadcs_amd import workloads
    long = workloads.markov(n, seed=5) if kind == "markov" else np.random.default_rng(5).integers(0, 256, n, dtype=np.uint8)
    texts = [long, workloads.protein(70_001, seed=6)]
    lengths = np.array([t.size for t in texts], dtype=np.int64)
    offsets, span = gpu.gpu_batch_layout(lengths)
    host = np.zeros(span + 64, dtype=np.uint8)
    for t, o in zip(texts, offsets.tolist()):
        host[o:o + t.size] = t
    print(f"{kind}: a batch of {span} bytes", flush=True)
    d_texts = gpu.DeviceBuffer.from_host(host)
    total = int(lengths.sum())
    d_sa, d_bwt = gpu.DeviceBuffer(4 * total), gpu.DeviceBuffer(total)
    with gpu.GpuContext(0, batch_lengths=lengths) as ctx:
        primaries = gpu.gpu_batch_build_device(ctx, d_texts.ptr, lengths, d_sa.ptr, d_bwt.ptr)
    at = 0
    for i, t in enumerate(texts):
        result = gpu.gpu_check_device(d_texts.ptr + int(offsets[i]), t.size, d_sa.ptr + 4 * at, d_bwt.ptr + at, int(primaries[i]))
        assert result == (0, -1), f"text {i} of {t.size} bytes"
        at += t.size
    for buffer in (d_texts, d_sa, d_bwt):
        buffer.free()
