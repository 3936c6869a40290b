"""Performance workloads of the framework: what a training job or a study has it do, through its public entry points.

A case is a dict of plain values; ``kind`` names the work and the other keys size it.  The kinds are the ways in which the
package is used:

  codec      the two (with ``fused`` three) codec calls on one vector: compress, ring step, decompress, through ``capi``
  ring       one rank's codec calls for one bucket in a compressed ring of ``world`` ranks: the compressor object's
             compression, dec_compression and decompression, in the order of the ring schedule
  stream     one training step of the dynamic-bitrate hook on one rank: every bucket through ``SinglePassBuckets``, then
             the search for the next step's offset on the histogram of the norms
  dynamic    one bucket of the dynamic-bitrate all-reduce with ``world`` ranks in one GPU's memory
  fixed      one bucket of the fixed-proportion all-reduce, likewise
  eden       EDEN's compress and decompress of one vector
  thc        THC's compress of one bucket and decompress of the aggregate
  rht        the blocked randomized Hadamard transform fused with the codec, there and back

``listed()`` takes its sizes from the repository's configurations (25 MB buckets of 6,553,600 elements, the ring of
8 x 124,439,808, 2^20 and 2^30 elements, the microbenchmark's 268,435,456) and adds small and ragged ones; ``draw(rng)``
gives further cases of the same kinds.
"""
import math

import torch

from dynamiq_sigcomm_artifact_amd import bitrate, capi, compressors, dynamiq_pipeline
from dynamiq_sigcomm_artifact_amd.eden import Eden
from dynamiq_sigcomm_artifact_amd.ring_sim import split_chunks
from dynamiq_sigcomm_artifact_amd.thc import OldINCACudaHadamardCompressor

DEVICE = "cuda:0"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
SUPERCHUNK = 256
TARGET_BITS = 4.375                 # the "5bit" method less the scales
BUCKET = 6553600                    # elements of a 25 MB bucket at 32 bits


def listed():
    return [
        # the last, small bucket of a model (norms and biases): eight ranks, seventeen short calls, all latency
        {"name": "ring_small_bucket", "kind": "ring", "n": 65792, "world": 8, "nbits": 4, "strategy": 2, "philox": False},
        # an ordinary bucket on a node of four, at the widest codes
        {"name": "ring_25mb_bucket", "kind": "ring", "n": BUCKET, "world": 4, "nbits": 8, "strategy": 3, "philox": False},
        # binary16 gradients of an odd length through the module's default strategy (flat scales)
        {"name": "codec_fp16_odd", "kind": "codec", "n": 1000016, "dtype": "fp16", "nbits": 4, "strategy": 0, "fused": False},
        # the headline: a 25 MB bucket of 32-bit gradients, compress and decompress
        {"name": "codec_25mb_fp32", "kind": "codec", "n": BUCKET, "dtype": "fp32", "nbits": 4, "strategy": 2, "fused": False},
        # the reference's microbenchmark: a bucket of half a gigabyte, with the fused ring step
        {"name": "codec_2p28_bf16", "kind": "codec", "n": 1 << 28, "dtype": "bf16", "nbits": 4, "strategy": 3, "fused": True},
        # a training step of a dynamic-bitrate hook: eight 25 MB buckets and a ragged last one
        {"name": "stream_step", "kind": "stream", "n": BUCKET, "buckets": 9, "last": 1234567, "strategy": 2, "streams": 2,
         "graphs": True},
        # a study of eight ranks on a short, ragged bucket
        {"name": "dynamic_w8_ragged", "kind": "dynamic", "n": 1000003, "world": 8, "strategy": 3},
        # the configuration of 8 x 124,439,808 gradients as one bucket
        {"name": "dynamic_w8_124m", "kind": "dynamic", "n": 124439808, "world": 8, "strategy": 2},
        # the fixed-proportion hook on two ranks, a bucket that ends inside a superchunk
        {"name": "fixed_w2_25mb", "kind": "fixed", "n": BUCKET - 77, "world": 2, "method": "5bit", "strategy": 2},
        # EDEN on 2^20 elements
        {"name": "eden_2p20", "kind": "eden", "n": 1 << 20, "dtype": "fp32", "nbits": 4},
        # THC on a 25 MB bucket, padded to the next power of two
        {"name": "thc_25mb", "kind": "thc", "n": BUCKET, "dtype": "fp32", "levels": 64, "nclients": 8},
        # rotation fused with the codec at the largest size in use
        {"name": "rht_2p30", "kind": "rht", "n": 1 << 30, "block": 8192, "nbits": 5},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("codec", "ring", "stream", "dynamic", "fixed", "eden", "thc", "rht"))
    if kind == "codec":
        dtype = rng.choice(("fp16", "bf16", "fp32"))
        strategy = rng.choice((0, 1, 2, 2, 3, 3) if dtype == "fp16" else (2, 3))
        unit = SUPERCHUNK if strategy >= 2 else 16
        return {"kind": kind, "n": -(-_log_uniform(rng, 4096, 1 << 27) // unit) * unit, "dtype": dtype,
                "nbits": rng.choice((2, 4, 5, 8)), "strategy": strategy, "fused": dtype != "fp16" and rng.random() < 0.5}
    if kind == "ring":
        return {"kind": kind, "n": -(-_log_uniform(rng, 1 << 15, 1 << 26) // SUPERCHUNK) * SUPERCHUNK,
                "world": rng.randint(2, 8), "nbits": rng.choice((2, 4, 5, 8)), "strategy": rng.choice((2, 3)),
                "philox": rng.random() < 0.3}
    if kind == "stream":
        n = _log_uniform(rng, 1 << 18, 2 * BUCKET)
        return {"kind": kind, "n": n, "buckets": rng.randint(2, 12), "last": rng.randint(n // 20, n), "strategy": rng.choice((2, 3)),
                "streams": rng.choice((1, 2, 2, 3)), "graphs": rng.random() < 0.7}
    if kind == "dynamic":
        return {"kind": kind, "n": _log_uniform(rng, 1 << 16, 1 << 25), "world": rng.randint(1, 8), "strategy": rng.choice((2, 3))}
    if kind == "fixed":
        return {"kind": kind, "n": _log_uniform(rng, 1 << 16, 1 << 25), "world": rng.randint(1, 4),
                "method": rng.choice(("3bit", "4bit", "5bit", "6bit", "7bit")), "strategy": rng.choice((2, 3))}
    if kind == "eden":
        return {"kind": kind, "n": _log_uniform(rng, 1 << 12, 1 << 24), "dtype": rng.choice(("fp32", "bf16")), "nbits": rng.choice((2, 4, 5, 8))}
    if kind == "thc":
        return {"kind": kind, "n": _log_uniform(rng, 1 << 12, 1 << 24), "dtype": rng.choice(("fp32", "bf16")),
                "levels": rng.choice((16, 64, 256)), "nclients": rng.choice((2, 4, 8))}
    block = 1 << rng.randint(10, 15)
    return {"kind": kind, "n": max(1, _log_uniform(rng, 1 << 19, 1 << 27) // block) * block, "block": block, "nbits": rng.choice((2, 4, 5, 8))}


# ---- inputs ------------------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _gradient(n, g, dtype):
    """heavy-tailed gradients: Student-t(3) * 1e-3, one entry in a thousand a hundred times as large"""
    x = torch.randn(n, generator=g, device=DEVICE)
    chi = torch.zeros(n, device=DEVICE)
    for _ in range(3):
        chi.add_(torch.randn(n, generator=g, device=DEVICE).square_())
    x.div_(chi.div_(3.0).sqrt_()).mul_(1e-3)
    x[torch.randint(0, n, (max(1, n // 1000),), generator=g, device=DEVICE)] *= 100.0
    return x.to(dtype)


def _layered(n, g, dtype, scale=1.0):
    """the gradients of a model's consecutive tensors: Gaussian, with a scale of its own (log-normal, sigma 1.5, around
    1e-3) for every run of 2^18 elements"""
    runs = -(-n // (1 << 18))
    x = torch.randn(n, generator=g, device=DEVICE)
    scales = torch.exp(torch.randn(runs, generator=g, device=DEVICE) * 1.5 + math.log(1e-3)) * scale
    return x.mul_(scales.repeat_interleave(1 << 18)[:n]).to(dtype)


def _offset(norms):
    """the offset of the width rule that meets the target on these norms: the search of the first compressed step"""
    return bitrate.dynamic_bitrate_binary_search_u(norms, TARGET_BITS)[0]


def _norms(x, world):
    nsc = -(-x.numel() // SUPERCHUNK)
    stats = torch.empty((nsc, 2), dtype=torch.bfloat16, device=DEVICE)
    capi.superchunk_stats(x, stats, None, x.numel(), world)
    return stats


def _codec_prepare(case, g):
    n, nbits, strategy, dtype = case["n"], case["nbits"], case["strategy"], DTYPES[case["dtype"]]
    size = capi.required_bytes(n, nbits, 16, strategy)
    s = {"src": _gradient(n, g, dtype),
         "pool": torch.rand(n, generator=g, device=DEVICE).to(torch.float16 if dtype == torch.float16 else torch.bfloat16),
         "packed": torch.zeros(size, dtype=torch.uint8, device=DEVICE), "out": torch.empty(n, dtype=dtype, device=DEVICE)}
    if case["fused"]:
        s["send"] = torch.zeros(size, dtype=torch.uint8, device=DEVICE)
        s["local"] = _gradient(n, g, dtype)
    return s


def _codec_run(case, s):
    n, nbits, strategy = case["n"], case["nbits"], case["strategy"]
    capi.scaling_compress(s["src"], s["packed"], s["pool"], n, nbits, 16, strategy)
    last = s["packed"]
    if case["fused"]:
        last = s["send"]
        capi.scaling_dec_comp(s["packed"], s["local"], last, s["pool"], n, nbits, 16, strategy)
    capi.scaling_decompress(last, s["out"], n, nbits, 16, strategy)
    return [s["packed"], last, s["out"]] if case["fused"] else [s["packed"], s["out"]]


def _codec_work(case):
    n, e = case["n"], DTYPES[case["dtype"]].itemsize
    p = capi.required_bytes(n, case["nbits"], 16, case["strategy"])
    passes = 3 if case["fused"] else 2
    return {"bytes": (e + 2) * n + p + ((e + 2) * n + 2 * p if case["fused"] else 0) + p + e * n, "flops": 8 * passes * n}


def _compressor(case, nbits, n, world, rank, g):
    cls = compressors.Mee_Dynamic_Range_GPU_kern if case["strategy"] == 3 else compressors.Aee_Dynamic_Range_GPU_kern
    params = {"d": {"bucket": n}, "world_size": world, "rank": rank}
    if case.get("philox"):
        params["philox_seed"] = 2026
    return cls(nbits, 16, params, device=DEVICE, generator=g)


def _ring_prepare(case, g):
    n, world = case["n"], case["world"]
    c = _compressor(case, case["nbits"], n, world, 0, g)
    vec, out = _gradient(n, g, torch.bfloat16), torch.empty(n, dtype=torch.bfloat16, device=DEVICE)
    chunks = split_chunks(vec, world, SUPERCHUNK)
    peer = _compressor(case, case["nbits"], n, world, 1, g)

    def received():
        buf = c.create_tensor(chunks[0], torch.uint8)
        peer.compression(_gradient(chunks[0].numel(), g, torch.bfloat16), buf)
        return buf

    return {"codec": c, "chunks": chunks, "out": out, "outs": split_chunks(out, world, SUPERCHUNK),
            "send": [c.create_tensor(chunks[0], torch.uint8) for _ in range(world)],
            "partial": [received() for _ in range(world - 1)], "final": [received() for _ in range(world - 1)]}


def _ring_run(case, s):
    world, c, chunks, outs, send = case["world"], s["codec"], s["chunks"], s["outs"], s["send"]
    # reduce-scatter: the own chunk first, then what the neighbour sent plus the local chunk; the last step's chunk is ours
    c.compression(chunks[0], send[0])
    for step in range(1, world):
        c.dec_compression(s["partial"][step - 1], chunks[-step], send[step])
    c.decompression(send[world - 1], outs[1 - world])
    # all-gather: the other ranks' reduced chunks
    for step in range(world - 1):
        c.decompression(s["final"][step], outs[-step])
    return [s["out"]] + send


def _ring_work(case):
    n, p = case["n"], capi.required_bytes(case["n"], case["nbits"], 16, case["strategy"])
    per = 1.0 - 1.0 / case["world"]
    pool = 0 if case["philox"] else 2
    return {"bytes": (2 + pool) * n + p + per * p + per * p + 2 * n, "flops": (8 + 8 * per + 8) * n}


def _stream_prepare(case, g):
    sizes = [case["n"]] * (case["buckets"] - 1) + [case["last"]]
    xs = [_layered(n, g, torch.bfloat16) for n in sizes]
    hist = bitrate.NormHistogram(DEVICE)
    hist.result[0] = _offset([_norms(x, 1)[:, 1] for x in xs])
    pipe = dynamiq_pipeline.SinglePassBuckets(DEVICE, strategy=case["strategy"], seed=3, streams=case["streams"], graphs=case["graphs"],
                                              u=hist.result[0:1], norm_histogram=hist)
    return {"pipe": pipe, "hist": hist, "pairs": [(x, torch.empty_like(x)) for x in xs]}


def _stream_run(case, s):
    pipe, hist = s["pipe"], s["hist"]
    pipe.begin_step()
    pipe.run_all(s["pairs"])
    pipe.join()
    hist.launch_search(1, hist.result[0:1], TARGET_BITS)
    return [out for _, out in s["pairs"]] + [hist.result]


def _stream_work(case):
    n = (case["buckets"] - 1) * case["n"] + case["last"]
    return {"bytes": 4 * n, "flops": 20 * n}


def _ranks(case, g):
    """one vector per rank, the ranks' scales spread over two decades"""
    world, base = case["world"], _layered(case["n"], g, torch.float32)
    spread = [10.0 ** (-1.0 + 2.0 * k / max(1, world - 1)) for k in range(world)]
    return [torch.randn(case["n"], generator=g, device=DEVICE).mul_(base).mul_(1e3 * s).to(torch.bfloat16) for s in spread]


def _dynamic_prepare(case, g):
    vecs, world = _ranks(case, g), case["world"]
    total = _norms(vecs[0], world)
    for v in vecs[1:]:
        total.add_(_norms(v, world))
    u = torch.full((1,), _offset([total[:, 1]]), dtype=torch.float64, device=DEVICE)
    return {"vecs": vecs, "u": u, "outs": [torch.empty_like(v) for v in vecs], "work": {}}


def _dynamic_run(case, s):
    outs, total, counts = dynamiq_pipeline.dynamic_bitrate_allreduce_single_pass(
        s["vecs"], s["u"], strategy=case["strategy"], seed=5, out=s["outs"], work=s["work"])
    return outs + [total, counts]


def _fixed_prepare(case, g):
    n, world = case["n"], case["world"]
    padded = -(-n // SUPERCHUNK) * SUPERCHUNK
    codecs = {q: [_compressor(case, q, padded, world, r, g) for r in range(world)] for q in (8, 4, 2)}
    vecs = _ranks(case, g)
    return {"vecs": vecs, "codecs": codecs, "thresholds": bitrate.fixed_proportion_thresholds(case["method"]),
            "outs": [torch.empty_like(v) for v in vecs]}


def _fixed_run(case, s):
    outs, total, order, _ = dynamiq_pipeline.fixed_proportion_allreduce_grouped(s["vecs"], s["thresholds"], s["codecs"], out=s["outs"])
    return outs + [total]


def _allreduce_work(case):
    n, world = case["n"], case["world"]
    return {"bytes": 4 * n * world, "flops": (6 + 8 * world) * n + 8 * n * world}


def _eden_prepare(case, g):
    return {"eden": Eden(device=DEVICE), "vec": _gradient(case["n"], g, DTYPES[case["dtype"]])}


def _eden_run(case, s):
    data = s["eden"].compress(s["vec"], case["nbits"], 42)
    out = s["eden"].decompress(data)
    return {"packed": [d["packed_bins"] for d in data], "scale": [d["scale"] for d in data], "out": out}


def _eden_work(case):
    n, e = case["n"], DTYPES[case["dtype"]].itemsize
    return {"bytes": 2 * e * n + 2 * n * case["nbits"] / 8.0, "flops": 2 * n * math.log2(n) + 12 * n}


def _thc_prepare(case, g):
    n, dim = case["n"], 1 << (case["n"] - 1).bit_length()
    key = (0, 0)
    codec = OldINCACudaHadamardCompressor({"d": {key: dim}, "size": {key: n}, "seed": 42, "T": 3.0, "device": DEVICE,
                                           "quantization_levels": case["levels"], "nclients": case["nclients"], "rank": 0})
    grad = _gradient(n, g, DTYPES[case["dtype"]])
    norm = grad.float().norm()
    total = torch.zeros(dim, dtype=torch.float32, device=DEVICE)
    for _ in range(case["nclients"]):
        total += codec.compress(_gradient(n, g, DTYPES[case["dtype"]]), key, norm).float()
    return {"codec": codec, "key": key, "grad": grad, "norm": norm, "total": total.to(torch.bfloat16)}


def _thc_run(case, s):
    levels = s["codec"].compress(s["grad"], s["key"], s["norm"])
    return [levels, s["codec"].decompress(s["total"], s["key"])]


def _thc_work(case):
    n, e = case["n"], DTYPES[case["dtype"]].itemsize
    dim = 1 << (n - 1).bit_length()
    return {"bytes": e * n + 4 * dim + 2 * dim + 2 * dim + 4 * n, "flops": 2 * dim * math.log2(dim) + 10 * dim}


def _rht_prepare(case, g):
    n, nbits = case["n"], case["nbits"]
    sign = torch.empty(n // 32, dtype=torch.int32, device=DEVICE)
    capi.rand_diag_bits(sign, n, 1234)
    return {"src": torch.randn(n, generator=g, device=DEVICE).mul_(1e-3), "sign": sign,
            "packed": torch.zeros(capi.required_bytes(n, nbits, 16, 2), dtype=torch.uint8, device=DEVICE),
            "out": torch.empty(n, dtype=torch.float32, device=DEVICE)}


def _rht_run(case, s):
    block, nbits, scale = case["block"], case["nbits"], 1.0 / math.sqrt(case["block"])
    capi.rht_scaling_compress(s["src"], s["sign"], s["packed"], block, scale, nbits, 2, seed=1, step=0)
    capi.scaling_decompress_irht(s["packed"], s["sign"], s["out"], block, scale, nbits, 2)
    return [s["packed"], s["out"]]


def _rht_work(case):
    n, p = case["n"], capi.required_bytes(case["n"], case["nbits"], 16, 2)
    return {"bytes": 8 * n + 2 * p + n / 4, "flops": 2 * n * math.log2(case["block"]) + 16 * n}


_KINDS = {
    "codec": (_codec_prepare, _codec_run, _codec_work),
    "ring": (_ring_prepare, _ring_run, _ring_work),
    "stream": (_stream_prepare, _stream_run, _stream_work),
    "dynamic": (_dynamic_prepare, _dynamic_run, _allreduce_work),
    "fixed": (_fixed_prepare, _fixed_run, _allreduce_work),
    "eden": (_eden_prepare, _eden_run, _eden_work),
    "thc": (_thc_prepare, _thc_run, _thc_work),
    "rht": (_rht_prepare, _rht_run, _rht_work),
}


def prepare(case, seed):
    return {"case": case, "state": _KINDS[case["kind"]][0](case, _generator(seed))}


def run(state):
    case = state["case"]
    return _KINDS[case["kind"]][1](case, state["state"])


def work(case):
    return _KINDS[case["kind"]][2](case)


def tolerance(case):
    """The codecs are defined to the bit: packed bytes, widths and decoded values.  EDEN's norm and scale are sums, and a
    rotated value that lies on a boundary of its table may go either way; THC's levels likewise."""
    if case["kind"] == "eden":
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-4}
    if case["kind"] == "thc":
        return {"rel": 1e-4, "max": 0.2}
    return "exact"
