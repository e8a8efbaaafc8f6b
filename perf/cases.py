"""The work that a program using sadcs_amd has it do, as cases that can be timed.

Every case is one kind of call at one size:

  device    a text resident on the GPU, outputs left there (gpu_build_device): a pipeline that
            indexes what it already holds on the device
  host      a text and outputs in host memory on a kept context (gpu_build): the command line's
            build and a library call from C++ or Python
  batch     many texts on the device in one construction (gpu_batch_build_device)
  documents many short texts from and to host memory in one construction (gpu_batch_build)
  serve     requests submitted to the continuous-batching server and waited for (Server)

Texts come from the generators of the benchmark's configurations (sadcs_amd.workloads): uniform
ACGT, DNA-like (repeats with substitutions, runs of N), order-3 Markov text over 96 printable
bytes, protein-like and periodic. Outputs are whole: the suffix array, the BWT, the primary index.
"""
import math
import random

import numpy as np
import torch

import sadcs_amd
from sadcs_amd import workloads

KiB, MiB = 1 << 10, 1 << 20


def listed():
    return [
        # The smallest requests: a short sequence or record, one call at a time. Latency only.
        {"name": "host_protein_4K", "call": "host", "text": "protein", "n": 4099, "cover": 32, "sa": True, "bwt": True},
        # The median served request (256 KiB), one at a time on a kept context.
        {"name": "host_dna_256K", "call": "host", "text": "dna_uniform", "n": 256 * KiB - 1, "cover": 32, "sa": True, "bwt": True},
        # A strongly repetitive text: one request in ten of the serving mix is periodic.
        {"name": "device_periodic_2M", "call": "device", "text": "periodic", "n": 2 * MiB + 77, "cover": 32, "sa": True, "bwt": True},
        # Only the BWT (a compressor's front end), protein-like, on the device.
        {"name": "device_bwt_protein_8M", "call": "device", "text": "protein", "n": 8 * MiB + 5, "cover": 32, "sa": False, "bwt": True},
        # 16 MiB of uniform ACGT at the mod-128 cover: the first single-text configuration.
        {"name": "device_dna_16M_c128", "call": "device", "text": "dna_uniform", "n": 16 * MiB, "cover": 128, "sa": True, "bwt": True},
        # Only the suffix array of a file's worth of text, pageable host memory both ways.
        {"name": "host_sa_markov_24M", "call": "host", "text": "markov", "n": 24 * MiB - 333, "cover": 32, "sa": True, "bwt": False},
        # A chromosome-sized DNA-like text at each cover: the second configuration.
        {"name": "device_dnalike_256M", "call": "device", "text": "dna_like", "n": 256 * MiB, "cover": 32, "sa": True, "bwt": True},
        {"name": "device_dnalike_256M_c128", "call": "device", "text": "dna_like", "n": 256 * MiB, "cover": 128, "sa": True, "bwt": True},
        # The headline: 1 GiB of Markov text, SA and BWT, resident on the device.
        {"name": "device_markov_1G", "call": "device", "text": "markov", "n": 1024 * MiB, "cover": 32, "sa": True, "bwt": True},
        # The batched configuration's mix (log-uniform lengths, DNA-like and Markov), a quarter of its texts.
        {"name": "batch_1024", "call": "batch", "count": 1024, "lo": 1 * KiB, "hi": 4 * MiB, "cover": 32, "sa": True, "bwt": True},
        # A page of short documents from host memory in one construction.
        {"name": "documents_512", "call": "documents", "count": 512, "lo": 200, "hi": 16 * KiB, "cover": 32, "sa": True, "bwt": True},
        # The serving configuration: a burst of mixed requests (lognormal, median 256 KiB).
        {"name": "serve_24", "call": "serve", "count": 24, "cover": 32, "sa": True, "bwt": True},
    ]


def _log_int(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    """One more case of the same ranges: 1 KiB to 256 MiB alone, batches up to 256 MiB, bursts."""
    call = rng.choice(["device", "device", "device", "host", "host", "batch", "documents", "serve"])
    cover = rng.choice([32, 32, 32, 128])
    sa, bwt = rng.choice([(True, True), (True, True), (True, False), (False, True)])
    if call in ("device", "host"):
        text = rng.choice(["dna_uniform", "dna_like", "markov", "protein", "periodic"])
        most = {"device": 256 * MiB, "host": 32 * MiB}[call]
        if cover == 128:
            most = min(most, 128 * MiB)
        if text == "periodic":
            most = min(most, 8 * MiB)
        return {"call": call, "text": text, "n": _log_int(rng, 1 * KiB, most), "cover": cover, "sa": sa, "bwt": bwt}
    if call == "batch":
        return {"call": call, "count": rng.randrange(2, 400), "lo": 1 * KiB, "hi": _log_int(rng, 16 * KiB, 2 * MiB),
                "cover": cover, "sa": sa, "bwt": bwt}
    if call == "documents":
        return {"call": call, "count": rng.randrange(20, 800), "lo": rng.randrange(1, 400), "hi": _log_int(rng, 1 * KiB, 64 * KiB),
                "cover": cover, "sa": sa, "bwt": bwt}
    return {"call": call, "count": rng.randrange(4, 40), "cover": 32, "sa": sa, "bwt": bwt}


# ---- inputs ---------------------------------------------------------------------------------------


def _text(case, seed):
    return getattr(workloads, case["text"])(case["n"], seed=seed)


def _documents(case, seed):
    """Short texts of log-uniform length (the same for every seed), alternating protein-like, Markov and ACGT."""
    rng = random.Random(case["count"])
    kinds = (workloads.protein, workloads.markov, workloads.dna_uniform)
    return [kinds[i % 3](_log_int(rng, case["lo"], case["hi"]), seed=seed * 1000 + i) for i in range(case["count"])]


def _request_lengths(case):
    """The serving mix: the first requests of one fixed stream, so that every seed offers the same load."""
    lengths, kinds = workloads.serving_requests(case["count"], seed=5, cap=16 * MiB)
    return lengths.tolist(), kinds.tolist()


def _requests(case, seed):
    return [workloads.serving_text(n, k, seed * 1000 + i) for i, (n, k) in enumerate(zip(*_request_lengths(case)))]


def _batch_lengths(case):
    """Log-uniform lengths in a mixed order, the same for every seed: up to 32 distinct lengths."""
    classes = min(32, case["count"])
    ratio = math.log(case["hi"] / case["lo"])
    lengths = [int(case["lo"] * math.exp(ratio * (i % classes + 0.5) / classes)) for i in range(case["count"])]
    random.Random(case["count"]).shuffle(lengths)
    return np.array(lengths, dtype=np.int64)


def _batch_text(case, seed, lengths, offsets, span):
    """Half DNA-like, half Markov texts (workloads.batch_buffer alternates them) at the layout's offsets."""
    out = np.zeros(span + 64, dtype=np.uint8)
    for k, n in enumerate(sorted(set(lengths.tolist()))):
        where = np.flatnonzero(lengths == n)
        buffer, starts, _ = workloads.batch_buffer(where.size, seed * 100 + k, n, n)
        for at, start in zip(offsets[where].tolist(), starts.tolist()):
            out[at:at + n] = buffer[start:start + n]
    return out


def _outputs(case, total):
    sa = torch.empty(total, dtype=torch.int32, device="cuda") if case["sa"] else None
    bwt = torch.empty(total, dtype=torch.uint8, device="cuda") if case["bwt"] else None
    return sa, bwt


def prepare(case, seed):
    state = {"case": case}
    if case["call"] == "device":
        n = case["n"]
        host = getattr(workloads, case["text"])(n, seed=seed, padding=64)
        state["text"] = torch.from_numpy(host).cuda()
        state["sa"], state["bwt"] = _outputs(case, n)
        state["context"] = sadcs_amd.GpuContext(n, cover=case["cover"])
    elif case["call"] == "host":
        state["text"] = _text(case, seed)
        state["context"] = sadcs_amd.GpuContext(case["n"], cover=case["cover"])
    elif case["call"] == "batch":
        lengths = _batch_lengths(case)
        offsets, span = sadcs_amd.gpu_batch_layout(lengths)
        host = _batch_text(case, seed, lengths, offsets, span)
        state["text"] = torch.from_numpy(host).cuda()
        state["lengths"] = lengths
        state["sa"], state["bwt"] = _outputs(case, int(lengths.sum()))
        state["context"] = sadcs_amd.GpuContext(0, cover=case["cover"], batch_lengths=lengths)
    elif case["call"] == "documents":
        state["texts"] = _documents(case, seed)
        state["context"] = sadcs_amd.GpuContext(0, cover=case["cover"], batch_lengths=[t.size for t in state["texts"]])
    else:
        state["texts"] = _requests(case, seed)
        state["server"] = sadcs_amd.Server(memory_budget=2048 * MiB, cover=case["cover"], suffix_array=case["sa"], bwt=case["bwt"])
    torch.cuda.synchronize()
    return state


# ---- one pass -------------------------------------------------------------------------------------


def _joined(results):
    """Outputs of many texts, one after another: suffix arrays, BWTs and primary indexes."""
    out = {"primary": np.array([-1 if r[2] is None else r[2] for r in results], dtype=np.int32)}
    if results[0][0] is not None:
        out["sa"] = np.concatenate([r[0] for r in results])
    if results[0][1] is not None:
        out["bwt"] = np.frombuffer(b"".join(r[1] for r in results), dtype=np.uint8)
    return out


def run(state):
    case = state["case"]
    if case["call"] == "device":
        sa, bwt = state["sa"], state["bwt"]
        primary = sadcs_amd.gpu_build_device(state["context"], state["text"].data_ptr(), case["n"],
                                             sa.data_ptr() if sa is not None else None, bwt.data_ptr() if bwt is not None else None)
        return {"sa": sa, "bwt": bwt, "primary": primary}
    if case["call"] == "batch":
        sa, bwt = state["sa"], state["bwt"]
        primaries = sadcs_amd.gpu_batch_build_device(state["context"], state["text"].data_ptr(), state["lengths"],
                                                     sa.data_ptr() if sa is not None else None, bwt.data_ptr() if bwt is not None else None)
        return {"sa": sa, "bwt": bwt, "primary": primaries}
    if case["call"] == "host":
        sa, bwt, primary = sadcs_amd.gpu_build(state["text"], case["sa"], case["bwt"], context=state["context"])
        return {"sa": sa, "bwt": None if bwt is None else np.frombuffer(bwt, dtype=np.uint8), "primary": primary}
    if case["call"] == "documents":
        return _joined(sadcs_amd.gpu_batch_build(state["texts"], case["sa"], case["bwt"], context=state["context"]))
    server = state["server"]
    ids = [server.submit(t) for t in state["texts"]]
    return _joined([server.wait(i)[:3] for i in ids])


def _lengths(case):
    if case["call"] in ("device", "host"):
        return [case["n"]]
    if case["call"] == "batch":
        return _batch_lengths(case).tolist()
    if case["call"] == "documents":
        rng = random.Random(case["count"])
        return [_log_int(rng, case["lo"], case["hi"]) for _ in range(case["count"])]
    return _request_lengths(case)[0]


def work(case):
    """Each text read once and each output written once (4 bytes a row of the suffix array, 1 of the BWT)."""
    total = sum(_lengths(case))
    return {"bytes": total * (1 + (4 if case["sa"] else 0) + (1 if case["bwt"] else 0)), "flops": 0}


# ---- the same outputs in numpy --------------------------------------------------------------------


def _suffix_array(text):
    """Prefix doubling with a stable argsort per round."""
    n = text.size
    rank = text.astype(np.int64) + 1
    h = 1
    while True:
        second = np.zeros(n, dtype=np.int64)
        second[:max(n - h, 0)] = rank[h:]
        key = rank * (n + 257) + second
        sa = np.argsort(key, kind="stable")
        head = np.concatenate(([True], key[sa][1:] != key[sa][:-1]))
        rank = np.empty(n, dtype=np.int64)
        rank[sa] = np.cumsum(head)
        if head.all():
            return sa
        h *= 2


def _one(text, case):
    sa = _suffix_array(text)
    bwt = None
    primary = -1
    if case["bwt"]:
        row = int(np.flatnonzero(sa == 0)[0])
        others = text[sa[sa != 0] - 1]
        bwt = np.concatenate((text[-1:], others))
        primary = row + 1
    return sa.astype(np.int32) if case["sa"] else None, bwt, primary


def exact(case, seed):
    """Up to 1.5 MB of text (a few seconds); larger cases have no value here."""
    if sum(_lengths(case)) > 1500000:
        return None
    if case["call"] in ("device", "host"):
        sa, bwt, primary = _one(_text(case, seed), case)
        return {"sa": sa, "bwt": bwt, "primary": primary}
    if case["call"] == "batch":
        lengths = _batch_lengths(case)
        offsets, span = sadcs_amd.gpu_batch_layout(lengths)
        host = _batch_text(case, seed, lengths, offsets, span)
        texts = [host[o:o + n] for o, n in zip(offsets.tolist(), lengths.tolist())]
    elif case["call"] == "documents":
        texts = _documents(case, seed)
    else:
        texts = _requests(case, seed)
    results = [_one(t, case) for t in texts]
    out = {"primary": np.array([r[2] for r in results], dtype=np.int32)}
    if case["sa"]:
        out["sa"] = np.concatenate([r[0] for r in results])
    if case["bwt"]:
        out["bwt"] = np.concatenate([r[1] for r in results])
    return out
